"""An fp8 MLP's two weight gradients as one split launch of the persistent kernel."""
import pytest
import torch

from trainium_frontier_them_bones_amd import ops

pytestmark = pytest.mark.gpu


# the fewest rows, ranges of unequal length, two to eight ranges, every CU with a tile and a fifth of them without
@pytest.mark.parametrize("M,d,F", [(6144, 768, 3072), (8320, 768, 3072), (16384, 768, 2048), (6144, 1024, 4096), (16384, 512, 2048)])
def test_two_weight_gradients_in_one_launch(M, d, F):
    dev = torch.device("cuda:0")
    g = torch.Generator(device=dev).manual_seed(M + F)
    fp8 = lambda n, dt: torch.randn(M, n, generator=g, device=dev).to(dt)
    x8, hq8 = fp8(d, torch.float8_e4m3fn), fp8(F, torch.float8_e4m3fn)
    dp8, dy8 = fp8(F, torch.float8_e5m2), fp8(d, torch.float8_e5m2)
    row = torch.zeros(16, device=dev)
    row[5], row[7], row[13] = 8.0, 0.5, 2.0                          # s_dy, s_dp, s_h
    bytes_ = [t.view(torch.uint8) for t in (x8, dp8, hq8, dy8)]
    want = (dp8.double().t() @ x8.double()).div(0.5 * 4.0), (dy8.double().t() @ hq8.double()).div(8.0 * 2.0)
    fc, proj = ops.mlp8_dw8(*bytes_, row, out_dtype=torch.float32)
    for got, w in zip((fc, proj), want):
        # every product is exact; M of them are added in fp32 (2^-24 a step at most, of partial sums no larger than a few of the result's rms)
        assert ((got.double() - w).norm() / w.norm()).item() < M ** 0.5 * 2 ** -24 * 4
    old = torch.randn(F, d, generator=g, device=dev), torch.randn(d, F, generator=g, device=dev)
    acc = tuple(t.clone() for t in old)
    ops.mlp8_dw8(*bytes_, row, dw_fc=acc[0], dw_proj=acc[1], accumulate=True, out_dtype=torch.float32)
    assert torch.equal(acc[0], old[0] + fc) and torch.equal(acc[1], old[1] + proj)
    for got, w in zip(ops.mlp8_dw8(*bytes_, row), (fc, proj)):
        assert torch.equal(got, w.bfloat16())                        # one rounding
