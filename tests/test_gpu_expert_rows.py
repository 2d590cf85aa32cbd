"""The experts' products over all rows in the persistent kernel and the launch that finishes what it leaves: the bits of the kernels that few rows take."""
import pytest
import torch

from trainium_frontier_them_bones_amd import _lib

pytestmark = pytest.mark.gpu


# part of a round; one round and a little, finished by the second launch; more than 0.3 of a second round; experts of one tile of 128 rows each; one
# expert; none between others; rows that nobody has at the end; tables longer than a wavefront's lanes; two k-tiles and more
@pytest.mark.parametrize("d,F,tiles,nobody", [(1024, 256, [33, 0, 31, 1, 7], 0), (1024, 512, [65, 64, 2], 3), (1024, 256, [40, 41, 43, 45], 5),
                                              (768, 256, [1] * 90, 0), (512, 768, [300], 1), (256, 256, [511, 0, 2], 70)])
def test_rows_of_experts(d, F, tiles, nobody):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(d + F + len(tiles))
    E, M = len(tiles), 128 * (sum(tiles) + nobody)
    owner = torch.tensor([e for e, t in enumerate(tiles) for _ in range(t)] + [-1] * nobody, dtype=torch.int32, device=dev)
    fp8 = lambda dt, *s: torch.randn(*s, generator=g, device=dev).to(dt)  # noqa: E731
    x8, dy8 = fp8(torch.float8_e4m3fn, M, d), fp8(torch.float8_e5m2, M, d)
    w8 = fp8(torch.float8_e4m3fn, E, 4, F * d)
    rows = 2.0 ** torch.randint(-3, 3, (E, 16), generator=g, device=dev).float()
    s = torch.cuda.current_stream().cuda_stream

    def run(a, b):
        n = b - a
        y, dx, r = (torch.full((n, w), float("nan"), device=dev, dtype=torch.bfloat16) for w in (d, d, F))
        h8, dp8, hq8 = (torch.zeros(n, F, device=dev, dtype=torch.uint8) for _ in range(3))
        p = lambda t: t.data_ptr()  # noqa: E731
        own = owner[a // 128:b // 128].contiguous()
        xa, ga = x8[a:b].contiguous(), dy8[a:b].contiguous()
        _lib.call("tfb_moe_mlp8_fwd", p(xa), p(w8), p(rows), p(own), p(y), p(r), p(h8), n, d, F, s)
        _lib.call("tfb_moe_mlp8_bwd_q", p(ga), p(r), p(w8), p(rows), p(own), p(dx), 0, p(dp8), p(hq8), 448.0, n, d, F, s)
        torch.cuda.synchronize()
        return y, dx

    got = run(0, M)
    for a in range(0, M, 1024):
        b = min(a + 1024, M)
        for whole, part in zip(got, run(a, b)):
            assert torch.equal(whole[a:b].view(torch.int16), part.view(torch.int16)), a
    mine = owner.repeat_interleave(128) >= 0
    assert all(bool(torch.isfinite(t[mine]).all()) for t in got)
