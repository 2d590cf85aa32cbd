"""The loss head where its arithmetic can go wrong."""
import pytest
import torch

pytestmark = pytest.mark.gpu
bf16 = torch.bfloat16


def _rows(dev, N, V, seed, std=3.0):
    g = torch.Generator().manual_seed(seed)
    x = (std * torch.randn(N, V, generator=g)).to(bf16)
    return x.to(dev), torch.randint(0, V, (N,), generator=g).to(dev)


@pytest.mark.parametrize("V", [64, 2048, 2056, 8192])
@pytest.mark.parametrize("cap", [0.0, 15.0])
@pytest.mark.parametrize("at", ["target", "elsewhere", "all"])
def test_a_nan_logit_reaches_the_loss_and_the_gradient(dev, V, cap, at):
    """A row that holds a NaN has the loss NaN and a gradient of NaN in every column, in each of the loss kernels; the other
    rows have what they have without it."""
    from trainium_frontier_them_bones_amd import ops
    x, t = _rows(dev, 5, V, V)
    bad = x.clone()
    if at == "all":
        bad[2] = float("nan")
    else:
        bad[2, t[2] if at == "target" else (t[2] + 1) % V] = float("nan")
    w = torch.ones(5, device=dev)

    def passes(x):
        rows, lse = ops.loss_fwd(x, t, cap, w)
        one = x.clone()
        rows1, _ = ops.loss_fwd_bwd(one, t, w, cap)
        tk, wk = torch.stack([t, (t + 3) % V]), torch.full((2, 5), 0.5, device=dev)
        rows2, lse2 = ops.loss_multi_fwd(x, tk, wk, cap, 0.1)
        return [rows, rows1, rows2], [ops.loss_bwd(x, t, lse, w, cap), one, ops.loss_multi_bwd(x, tk, wk, lse2, w, cap, 0.1)]

    others = torch.tensor([0, 1, 3, 4], device=dev)
    for got, want in zip(passes(bad), passes(x)):
        for a, b in zip(got, want):
            assert bool(a[2].isnan().all()) and torch.equal(a[others], b[others]) and bool(b.isfinite().all())


@pytest.mark.parametrize("cap", [0.0, 15.0])
@pytest.mark.parametrize("N,V", [(128, 1024), (4096, 8192)])
def test_a_nan_activation_reaches_the_loss_head(dev, N, V, cap):
    """Training and evaluation of the LM head agree that a row with a NaN has no loss (the second size takes the persistent
    GEMM and a pass over its logits, the first the log-sum-exp in the GEMM's epilogue)."""
    from trainium_frontier_them_bones_amd import autograd as A
    g = torch.Generator().manual_seed(N)
    x = torch.randn(N, 128, generator=g).to(bf16).to(dev)
    x[3, 5] = float("nan")
    W = (0.05 * torch.randn(V, 128, generator=g)).to(bf16).to(dev).requires_grad_(True)
    t = torch.randint(0, V, (N,), generator=g).to(dev)
    loss = A.LmHeadLossFn.apply(x, W, t, cap, "mean")
    (gw,) = torch.autograd.grad(loss, W)
    with torch.no_grad():
        ev = A.LmHeadLossFn.apply(x, W, t, cap, "mean")
    assert bool(loss.isnan()) and bool(ev.isnan()) and bool(gw.isnan().any())
