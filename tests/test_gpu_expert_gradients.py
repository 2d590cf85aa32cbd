"""The experts' fp8 weight gradients, both of every expert in one launch."""
import pytest
import torch

from trainium_frontier_them_bones_amd import _lib

pytestmark = pytest.mark.gpu


# segments without rows (first, last, in the middle), of one tile and of two, equal ones; one expert, as many as there are lanes; tiles that the
# XCDs share evenly and not; the last row of the buffer the last of a segment
@pytest.mark.parametrize("d,F,tiles", [(256, 256, [1]), (256, 512, [0, 1, 2, 0, 3, 0]), (512, 768, [5, 5, 1, 5]), (1024, 2816, [0, 20, 1, 7]),
                                       (256, 256, [1, 2] * 32), (768, 256, [3, 0, 0, 9])])
@pytest.mark.parametrize("f32,accumulate", [(1, 0), (1, 1), (0, 0), (0, 1)])
def test_expert_gradients(d, F, tiles, f32, accumulate):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(d + F + len(tiles))
    E, M = len(tiles), 128 * sum(tiles)
    seg = torch.tensor([0] + tiles, device=dev).cumsum(0).mul(128).int()
    fp8 = lambda n, dt: torch.randn(M, n, generator=g, device=dev).to(dt)
    x8, hq8 = fp8(d, torch.float8_e4m3fn), fp8(F, torch.float8_e4m3fn)
    dp8, dy8 = fp8(F, torch.float8_e5m2), fp8(d, torch.float8_e5m2)
    rows = torch.ones(E, 16, device=dev)
    rows[:, 5], rows[:, 7], rows[:, 13] = 8.0, 2.0 ** torch.arange(E, device=dev).remainder(5), 0.5
    dt = torch.float32 if f32 else torch.bfloat16
    fc, proj = (torch.randn(E, *s, generator=g, device=dev).to(dt) for s in ((F, d), (d, F)))
    old = fc.clone(), proj.clone()
    assert x8.numel() == dy8.numel() == M * d and hq8.numel() == dp8.numel() == M * F and fc.numel() == proj.numel() == E * d * F
    _lib.call("tfb_moe_dw8", x8.data_ptr(), dp8.data_ptr(), hq8.data_ptr(), dy8.data_ptr(), rows.data_ptr(), 4.0, seg.data_ptr(), fc.data_ptr(),
              proj.data_ptr(), E, d, F, f32, accumulate, torch.cuda.current_stream().cuda_stream)
    for e in range(E):
        a, b = int(seg[e]), int(seg[e + 1])
        for got, was, (q, p), scale in ((fc, old[0], (dp8, x8), 4.0 * float(rows[e, 7])), (proj, old[1], (dy8, hq8), 4.0)):
            want = q[a:b].double().t() @ p[a:b].double() / scale
            if accumulate:
                want = want + was[e].double()
            # exact products, added in fp32 (by the matrix unit in blocks: 2^-16 of the norm covers its alignment), then one rounding to bf16
            tol = 2 ** -16 + (0 if f32 else 2 ** -9)
            assert ((got[e].double() - want).norm() <= tol * want.norm() + 1e-30).item()


# few rows per expert: a launch of the 128 x 128 kernel for each gradient. No rows, one k-tile and more, all of 16 experts, the last row of the
# buffer the last of a segment
@pytest.mark.parametrize("d,F,tiles", [(256, 256, [1]), (256, 256, [4, 4]), (256, 512, [2, 0, 3, 2]), (512, 1024, [1] * 8), (1024, 2816, [1, 2, 0, 1, 1, 1, 1, 1]),
                                       (256, 512, [1, 0] * 8)])
@pytest.mark.parametrize("f32,accumulate", [(1, 0), (0, 1)])
def test_one_launch_gives_the_bits_of_two(d, F, tiles, f32, accumulate):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(d + F + len(tiles))
    E, M = len(tiles), 128 * sum(tiles)
    seg = torch.tensor([0] + tiles, device=dev).cumsum(0).mul(128).int()
    fp8 = lambda n, dt: torch.randn(M, n, generator=g, device=dev).to(dt)  # noqa: E731
    x8, hq8 = fp8(d, torch.float8_e4m3fn), fp8(F, torch.float8_e4m3fn)
    dp8, dy8 = fp8(F, torch.float8_e5m2), fp8(d, torch.float8_e5m2)
    rows = torch.ones(E, 16, device=dev)
    dt = torch.float32 if f32 else torch.bfloat16
    old = [torch.randn(E, *s, generator=g, device=dev).to(dt) for s in ((F, d), (d, F))]
    assert x8.numel() == dy8.numel() == M * d and hq8.numel() == dp8.numel() == M * F
    out = []
    for rmax in (0, 128 * E):   # not known: one launch; some row for each expert: two
        assert _lib.lib().tfb_moe_dw8_one_launch_applies(E, d, F, rmax) == (rmax > 0)
        fc, proj = (t.clone() for t in old)
        _lib.call("tfb_moe_dw8_rows", x8.data_ptr(), dp8.data_ptr(), hq8.data_ptr(), dy8.data_ptr(), rows.data_ptr(), 4.0, seg.data_ptr(), fc.data_ptr(),
                  proj.data_ptr(), E, d, F, f32, accumulate, rmax, torch.cuda.current_stream().cuda_stream)
        out.append((fc, proj))
    assert torch.equal(out[0][0], out[1][0]) and torch.equal(out[0][1], out[1][1])
