"""The experts' up-projection and dH over all rows in the kernel that keeps the weights in registers: the bytes of the kernels that few rows take."""
import pytest
import torch

from trainium_frontier_them_bones_amd import _lib

pytestmark = pytest.mark.gpu


# experts of one tile and of none; an eighth of the rows that begins inside a tile; every tile another expert's; rows that nobody has, within
# an eighth and more than one; one expert; more tiles an eighth than a wavefront has lanes
@pytest.mark.parametrize("d,F,tiles,nobody", [(1024, 2816, [65, 0, 62, 1, 14, 46], 0), (768, 3072, [1] * 172, 0), (1024, 2816, [1] * 189, 1),
                                              (1024, 2816, [80, 70, 33], 7), (768, 3072, [100, 60], 37), (768, 3072, [173], 0),
                                              (768, 768, [300, 0, 200, 1, 150], 40), (1024, 768, [3, 690], 2)])
def test_up_and_dh_of_experts(d, F, tiles, nobody):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(d + F + len(tiles))
    E, M = len(tiles), 128 * (sum(tiles) + nobody)
    assert F // 256 * (M // 64) >= 16 * torch.cuda.get_device_properties(0).multi_processor_count
    owner = torch.tensor([e for e, t in enumerate(tiles) for _ in range(t)] + [-1] * nobody, dtype=torch.int32, device=dev)
    fp8 = lambda dt, *s: torch.randn(*s, generator=g, device=dev).to(dt)  # noqa: E731
    x8, dy8 = fp8(torch.float8_e4m3fn, M, d), fp8(torch.float8_e5m2, M, d)
    w8 = fp8(torch.float8_e4m3fn, E, 4, F * d)
    rows = 2.0 ** torch.randint(-3, 3, (E, 16), generator=g, device=dev).float()
    rows[::3] *= 1.1  # (scales that are no powers of two take the epilogues' general paths)
    s = torch.cuda.current_stream().cuda_stream

    def run(a, b):
        n = b - a
        y, dx, r = (torch.full((n, w), 7.0, device=dev, dtype=torch.bfloat16) for w in (d, d, F))
        h8, dp8, hq8 = (torch.full((n, F), 3, device=dev, dtype=torch.uint8) for _ in range(3))
        p = lambda t: t.data_ptr()  # noqa: E731
        own = owner[a // 128:b // 128].contiguous()
        xa, ga = x8[a:b].contiguous(), dy8[a:b].contiguous()
        _lib.call("tfb_moe_mlp8_fwd", p(xa), p(w8), p(rows), p(own), p(y), p(r), p(h8), n, d, F, s)
        _lib.call("tfb_moe_mlp8_bwd_q", p(ga), p(r), p(w8), p(rows), p(own), p(dx), 0, p(dp8), p(hq8), 448.0, n, d, F, s)
        torch.cuda.synchronize()
        return [t.view(torch.uint8).reshape(n, -1) for t in (r, h8, dp8, hq8, y, dx)]

    whole = run(0, M)
    for a in range(0, M, 1024):
        b = min(a + 1024, M)
        for name, t, part in zip(("r", "h8", "dp8", "hq8", "y", "dx"), whole, run(a, b)):
            assert torch.equal(t[a:b], part), (name, a)
    assert bool((whole[1][owner.repeat_interleave(128) < 0] == 3).all())  # (what nobody has is not written)
