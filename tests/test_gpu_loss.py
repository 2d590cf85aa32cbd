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


@pytest.mark.parametrize("cap", [7.0, 15.0, 30.0])
@pytest.mark.parametrize("std", [0.5, 2.0])
@pytest.mark.parametrize("N,V", [(128, 8192), (9600, 8192)])
def test_lse_of_evaluation_is_as_exact_as_that_of_training(dev, N, V, std, cap):
    """The log-sum-exp that evaluation takes in its GEMM's epilogue (first size) and in a pass over the logits (second) has no
    larger error against float64, on the logits it returned, than the training kernels' with their exact tanh: in the mean
    over the rows, where a bias of the terms stays and roundings cancel, and in the root mean square. The allowance of a
    tenth of an ulp of lse (2^-20 to 2^-19 here) is what the sums' different order and 128 rows leave of chance."""
    from trainium_frontier_them_bones_amd import ops
    g = torch.Generator().manual_seed(V + int(cap))
    d = 256
    x = torch.randn(N, d, generator=g).to(bf16).to(dev)
    W = (std / d ** 0.5 * torch.randn(V, d, generator=g)).to(bf16).to(dev)
    t = torch.randint(0, V, (N,), generator=g).to(dev)
    logits, _, lse = ops.lmhead_fwd(x, W, t, cap)
    _, plain = ops.loss_fwd(logits, t, cap)
    want = torch.cat([torch.logsumexp(cap * torch.tanh(part.double() / cap), -1) for part in logits.split(1024)])
    e, p = lse.double() - want, plain.double() - want
    ulp = 2.0 ** (torch.floor(torch.log2(want.mean())).item() - 23)
    print("cap %g std %g rows %d: mean %.3g rms %.3g, training's %.3g %.3g, ulp %.3g"
          % (cap, std, N, e.mean(), e.square().mean().sqrt(), p.mean(), p.square().mean().sqrt(), ulp))
    assert abs(e.mean()) < abs(p.mean()) + 0.1 * ulp
    assert e.square().mean().sqrt() < p.square().mean().sqrt() + 0.1 * ulp


@pytest.mark.parametrize("cap", [None, 15.0])
def test_fused_loss_node_gives_the_rows(dev, cap):
    """FusedLossFn.apply(logits, targets, softcap) is the loss of every row, ReducedLossFn their mean or sum."""
    from trainium_frontier_them_bones_amd import autograd as A, ops
    x, t = _rows(dev, 9, 264, 5)
    t[4] = -1
    want, _ = ops.loss_fwd(x, t, cap)
    rows = A.FusedLossFn.apply(x, t, cap)
    assert rows.shape == (9,) and torch.equal(rows, want)
    assert torch.allclose(A.ReducedLossFn.apply(x, t, False, cap), want.sum(), rtol=1e-6)
    assert torch.allclose(A.ReducedLossFn.apply(x, t, True, cap), want.sum() / 8, rtol=1e-6)
    a, b = x.clone().requires_grad_(True), x.clone().requires_grad_(True)
    (ga,) = torch.autograd.grad(A.FusedLossFn.apply(a, t, cap).sum(), a)
    (gb,) = torch.autograd.grad(A.ReducedLossFn.apply(b, t, False, cap), b)
    assert torch.equal(ga, gb)


def test_the_switch_for_the_one_pass_loss_head(dev, monkeypatch):
    """autograd.LM_HEAD_ONE_PASS = False takes the loss and its gradient in two passes: other launches, the same values."""
    from trainium_frontier_them_bones_amd import _lib, autograd as A
    g = torch.Generator().manual_seed(8)
    x = torch.randn(128, 128, generator=g).to(bf16).to(dev).requires_grad_(True)
    W = (0.05 * torch.randn(1024, 128, generator=g)).to(bf16).to(dev).requires_grad_(True)
    t = torch.randint(0, 1024, (128,), generator=g).to(dev)

    def step():
        rec = []
        _lib.TIMED["*"] = rec
        try:
            loss = A.LmHeadLossFn.apply(x, W, t, 15.0, "mean")
            grads = torch.autograd.grad(loss, (x, W))
        finally:
            del _lib.TIMED["*"]
        return loss.item(), grads, {r[2] for r in rec}

    one, grads1, names1 = step()
    monkeypatch.setattr(A, "LM_HEAD_ONE_PASS", False)
    two, grads2, names2 = step()
    assert "tfb_loss_fwd_bwd" in names1 and "tfb_loss_fwd_bwd" not in names2
    assert {"tfb_lmhead_fwd", "tfb_loss_bwd"} <= names2
    assert abs(one - two) < 1e-6 * one
    for a, b in zip(grads1, grads2):
        assert (a.float() - b.float()).norm() < 5e-3 * b.float().norm()


@pytest.mark.parametrize("cap", [0.5, 7.0, 15.0, 30.0, 50.0])
def test_tanh_has_the_bits_of_an_ieee_division(dev, cap):
    """The gradient factor 1 - tanh^2 of every bf16 bit pattern, each the target of a row of its own, with the kernels'
    reciprocal and with a division in the same fp32 expressions (NaN where the logit is one)."""
    from trainium_frontier_them_bones_amd import ops
    x = torch.arange(65536, dtype=torch.int32, device=dev).to(torch.int16).view(bf16)
    z = torch.zeros(65536, 8, dtype=bf16, device=dev)
    z[:, 3] = x
    t = torch.full((65536,), 3, device=dev)
    lse = torch.full((65536,), cap + 200.0, device=dev)              # no softmax left: -1 at the target, 0 elsewhere
    got = ops.loss_bwd(z, t, lse, torch.ones(65536, device=dev), cap)
    y = x.float() * (1.0 / torch.tensor(cap, device=dev))
    th = 1.0 - 2.0 / (torch.exp2(y * 2.8853900817779268) + 1.0)
    want = (-(1.0 - th * th)).to(bf16)
    nan = x.isnan()
    assert bool(got[nan, 3].isnan().all()) and torch.equal(got[~nan, 3], want[~nan])
    assert not bool(got[~nan][:, [0, 1, 2, 4, 5, 6, 7]].any())
