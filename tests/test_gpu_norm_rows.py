"""RMSNorm and its gradient at the edges of a row's lanes and of a grid: rows of one chunk to the widest, a row alone, a last workgroup
that is not full, and more workgroups than there are partial sums."""
import pytest
import torch

from trainium_frontier_them_bones_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("C", [8, 256, 512, 768, 776, 1024, 1032, 2048, 4096])
@pytest.mark.parametrize("rows", [1, 9, 4099])
@pytest.mark.parametrize("gain", [False, True])
@pytest.mark.parametrize("skip", [False, True])
def test_norm_pair(rows, C, gain, skip):
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(rows * C)
    x, gy, gs = (torch.randn(rows, C, generator=g).bfloat16() for _ in range(3))
    w = (1 + 0.2 * torch.randn(C, generator=g)).bfloat16() if gain else None
    to = lambda t: None if t is None else t.to(dev)
    eps = 1e-6
    s, y, inv = ops.rmsnorm_fwd(to(x), to(w), eps, to(gs) if skip else None)
    xs = (x.float() + gs.float()).bfloat16() if skip else x
    if skip:
        assert torch.equal(s.cpu(), xs)
    xd = xs.double()
    ref_inv = (xd.square().mean(1) + eps).rsqrt()
    ref = xd * ref_inv[:, None] * (1.0 if w is None else w.double())
    # the sum of C squares in fp32 is off by C / 2 roundings at most (of 2^-24 each), an output by one to bf16
    tol = 2.0**-8
    assert bool(((y.cpu().double() - ref).abs() <= tol * ref.abs()).all())
    assert bool(((inv.cpu().double() - ref_inv).abs() <= (C / 4 + 4) * 2.0**-24 * ref_inv).all())
    dx, dw, am = ops.rmsnorm_bwd(to(gy), to(xs), inv, to(w), to(gs) if skip else None, want_amax=True)
    again = ops.rmsnorm_bwd(to(gy), to(xs), inv, to(w), to(gs) if skip else None)
    assert torch.equal(dx, again[0]) and float(am.max()) == float(dx.abs().max())
    gh = gy.double() * (1.0 if w is None else w.double())
    dot = (gh * xd).sum(1, keepdim=True)
    i2 = ref_inv[:, None]
    rdx = i2 * (gh - xd * dot * i2 * i2 / C) + (gs.double() if skip else 0.0)
    # one rounding to bf16; before it fp32 terms of the size of inv |gh|, inv^3 |s| sum |gh s| / C and |gs|
    big = i2 * (gh.abs() + xd.abs() * (gh * xd).abs().sum(1, keepdim=True) * i2 * i2 / C) + gs.double().abs()
    assert bool(((dx.cpu().double() - rdx).abs() <= tol * rdx.abs() + (C / 4 + 8) * 2.0**-24 * big).all())
    if gain:
        rdw = (gy.double() * xd * i2).sum(0)
        bound = (gy.double() * xd * i2).abs().sum(0)
        assert bool(((dw.cpu().double() - rdw).abs() <= (rows / 8 + 64) * 2.0**-24 * bound).all())
    else:
        assert dw is None
