"""The experts' products over all rows with tiles of rows that nobody has between the experts': the bytes of the kernels that few rows take."""
import pytest
import torch

from trainium_frontier_them_bones_amd import _lib

pytestmark = pytest.mark.gpu


# (expert, tiles) in turn, -1: nobody's. A gap longer than half the table, with little in front of it and little behind; one tile of each in turn;
# gaps around an expert that comes twice, at the table's ends too
@pytest.mark.parametrize("runs", [[(0, 10), (-1, 400), (1, 100), (-1, 201)], [(0, 1), (-1, 1), (1, 1), (-1, 1)] * 178, [(-1, 3), (2, 300), (-1, 70), (0, 64), (-1, 130), (2, 140), (-1, 4)]])
@pytest.mark.parametrize("d,F", [(768, 768), (1024, 768)])
def test_gaps_between_experts(d, F, runs):
    dev = torch.device("cuda:0")
    table = [e for e, t in runs for _ in range(t)]
    E, M = 3, 128 * len(table)
    assert F // 256 * (M // 64) >= 16 * torch.cuda.get_device_properties(0).multi_processor_count and len(table) <= 800
    owner = torch.tensor(table, dtype=torch.int32, device=dev)
    g = torch.Generator(device=dev).manual_seed(d + len(runs))
    fp8 = lambda dt, *s: torch.randn(*s, generator=g, device=dev).to(dt)  # noqa: E731
    x8, dy8 = fp8(torch.float8_e4m3fn, M, d), fp8(torch.float8_e5m2, M, d)
    w8 = fp8(torch.float8_e4m3fn, E, 4, F * d)
    rows = 2.0 ** torch.randint(-3, 3, (E, 16), generator=g, device=dev).float()
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
    for a in range(0, M, 2048):
        b = min(a + 2048, M)
        for name, t, part in zip(("r", "h8", "dp8", "hq8", "y", "dx"), whole, run(a, b)):
            assert torch.equal(t[a:b], part), (name, a)
    assert bool((whole[1][owner.repeat_interleave(128) < 0] == 3).all())  # (what nobody has is not written)
