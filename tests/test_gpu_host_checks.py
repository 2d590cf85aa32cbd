"""What the native host layer refuses before a kernel is launched on it: operands and buffers that a kernel would read or
write out of range."""
import pytest
import torch

pytestmark = pytest.mark.gpu
bf16 = torch.bfloat16


def _t(dev, *shape, dtype=bf16, grad=False):
    return (0.05 * torch.randn(*shape, generator=torch.Generator().manual_seed(len(shape)))).to(dtype).to(dev).requires_grad_(grad)


def _calls(dev):
    """name -> (loss of the weights, weights): every node that adds a weight's gradient into its buffer."""
    from trainium_frontier_them_bones_amd import autograd as A
    from oracle import attention as O
    x = _t(dev, 256, 256, grad=True)
    w = [_t(dev, 256, 256, grad=True) for _ in range(2)]
    wf, wp = _t(dev, 512, 256, grad=True), _t(dev, 256, 512, grad=True)
    tg = torch.arange(256, device=dev)
    gain = _t(dev, 256, grad=True)
    cos, sin = (t.to(dev) for t in O.rope_tables(256, 64))
    wq = _t(dev, 768, 256, grad=True)
    emb = _t(dev, 128, 256, grad=True)
    router, ef, ep = _t(dev, 4, 256, dtype=torch.float32, grad=True), _t(dev, 4, 512, 256, grad=True), _t(dev, 4, 256, 512, grad=True)

    def fp8(cls, dw, *ws):
        st = cls(dw_fp8=dw)
        st.refresh(*ws)
        return st

    out = {
        "linear": (lambda: A.LinearFn.apply(x, w[0]).sum(), w[:1]),
        "linear8": (lambda: A.Linear8Fn.apply(x, w[1], fp8(A.Linear8State, False, w[1]), 4.0).sum(), w[1:]),
        "linear8 fp8": (lambda: A.Linear8Fn.apply(x, w[1], fp8(A.Linear8State, True, w[1]), 4.0).sum(), w[1:]),
        "qkv": (lambda: A.QkvRopeAttentionFn.apply(x.view(1, 256, 256), wq, cos, sin, 4, 0.125).sum(), [wq]),
        "mlp": (lambda: A.MlpFusedFn.apply(x, wf, wp).sum(), [wf, wp]),
        "mlp8": (lambda: A.Mlp8Fn.apply(x, wf, wp, fp8(A.Mlp8State, False, wf, wp)).sum(), [wf, wp]),
        "mlp8 fp8": (lambda: A.Mlp8Fn.apply(x, wf, wp, fp8(A.Mlp8State, True, wf, wp)).sum(), [wf, wp]),
        "head": (lambda: A.LmHeadLossFn.apply(x, w[0], tg, 0.0, "mean"), w[:1]),
        "norm": (lambda: A.RMSNormFn.apply(x, gain, 1e-6).sum(), [gain]),
        "norm pass": (lambda: A.RMSNormPassFn.apply(x, gain, 1e-6)[1].sum(), [gain]),
        "add norm": (lambda: A.AddRMSNormFn.apply(x, x, gain, 1e-6)[1].sum(), [gain]),
        "embedding": (lambda: A.EmbeddingFn.apply(tg % 128, emb).sum(), [emb]),
    }
    for name, dw in (("moe", False), ("moe fp8", True)):
        st = fp8(A.Moe8State, dw, ef, ep)
        out[name] = (lambda st=st: A.MoeMlp8Fn.apply(x, router, ef, ep, st, 2, None).sum(), [ef, ep])
    out["moe bf16"] = (lambda: A.MoeMlp8Fn.apply(x, router, ef, ep, None, 2, None).sum(), [ef, ep])
    out["router"] = (lambda: A.MoeMlp8Fn.apply(x, router, ef, ep, None, 2, None).sum(), [router])
    return out


FLAT = ("norm", "norm pass", "add norm", "embedding", "router")     # fp32 buffers of the weight's number of elements
BAD = {
    "too small": lambda w: torch.zeros((w.shape[0] // 2,) + tuple(w.shape[1:]), device=w.device),
    "too large": lambda w: torch.zeros((w.shape[0] * 2,) + tuple(w.shape[1:]), device=w.device),
    "strided": lambda w: torch.zeros(tuple(w.shape) + (2,), device=w.device)[..., 0],
    "fp16": lambda w: torch.zeros(w.shape, device=w.device, dtype=torch.float16),
    "fp64": lambda w: torch.zeros(w.shape, device=w.device, dtype=torch.float64),
    "on the host": lambda w: torch.zeros(w.shape),
    "no tensor": lambda w: [0.0],
}


def test_gradient_buffers_are_checked(dev):
    """A gradient buffer that a kernel would overrun, or fill as what it is not, is refused and left alone; a good one is
    filled with the gradient that autograd gets without it."""
    for name, (loss, ws) in _calls(dev).items():
        print(name, flush=True)
        plain = torch.autograd.grad(loss(), ws)
        for kind, make in BAD.items():
            for w in ws:
                w.grad_buf = make(w)
            with pytest.raises((RuntimeError, TypeError, ValueError)):
                loss().backward()
            for w in ws:
                if torch.is_tensor(w.grad_buf):
                    assert not bool(w.grad_buf.any()), (name, kind)
                    assert getattr(w, "grad_fresh", True), (name, kind)
        for dtype in (torch.float32,) if name in FLAT else (torch.float32, bf16):
            for w in ws:
                w.grad, w.grad_buf, w.grad_fresh = None, torch.full(w.shape, 7.0, device=dev, dtype=dtype), True
            loss().backward()
            for w, g in zip(ws, plain):
                assert w.grad is None and not w.grad_fresh
                assert (w.grad_buf.float() - g.float()).norm() < 5e-3 * g.float().norm(), (name, dtype)
        for w in ws:
            del w.grad_buf, w.grad_fresh


def test_a_buffer_for_the_norm_gradients_partial_sums_is_checked(dev):
    from trainium_frontier_them_bones_amd import autograd as A, ops
    x, w = _t(dev, 256, 256, grad=True), _t(dev, 256, grad=True)
    nb = ops.norm_bwd_blocks(256)
    w.dw_part = torch.zeros(nb - 1, 256, device=dev)
    with pytest.raises(ValueError):
        A.RMSNormFn.apply(x, w, 1e-6).sum().backward()
    w.dw_part = torch.zeros(nb, 256, device=dev)
    A.RMSNormFn.apply(x, w, 1e-6).sum().backward()
    assert bool(w.dw_part.any()) and w.grad is None


def test_operands_in_another_shape_give_the_same_results(dev):
    """Residuals, the embedding stream and the skip given as [B, T, H, D] or as rows, or strided: outputs have x's leading shape,
    values and gradients are those of the same operand in x's own shape, each gradient in its operand's shape."""
    from trainium_frontier_them_bones_amd import autograd as A, train_api as api
    B, T, C = 2, 128, 256
    l = [torch.tensor([v], device=dev) for v in (1.0, 0.3, 0.5)]
    w, wf, wp = _t(dev, C, C), _t(dev, 512, C), _t(dev, C, 512)
    st8, st = A.Linear8State(), A.Mlp8State()
    st8.refresh(w), st.refresh(wf, wp)
    calls = [lambda x, r: api.tail_norm2(x, r), lambda x, r: (api.final_norm(x, r),), lambda x, r: api.block_head(x, r, l[0], l[1]),
             lambda x, r: api.head_skip(x, r, r, *l), lambda x, r: (A.LinearFn.apply(x, w, r),),
             lambda x, r: (A.Linear8Fn.apply(x, w, st8, 4.0, None, r),), lambda x, r: (A.Mlp8Fn.apply(x, wf, wp, st, None, r),)]
    g = torch.Generator().manual_seed(3)
    x0, r0, gy = (torch.randn(B, T, C, generator=g).to(bf16).to(dev) for _ in range(3))
    for i, call in enumerate(calls):
        want = None
        for make in (lambda r: r.clone(), lambda r: r.view(B, T, 4, 64).clone(), lambda r: r.view(B * T, C).clone(),
                     lambda r: r.transpose(1, 2).contiguous().transpose(1, 2)):
            x, r = x0.clone().requires_grad_(True), make(r0).requires_grad_(True)
            out = call(x, r)
            assert all(o.shape == x.shape for o in out), i
            got = [o.detach() for o in out] + list(torch.autograd.grad(out, (x, r), [gy] * len(out)))
            assert got[-1].shape == r.shape
            got[-1] = got[-1].reshape(B, T, C)
            want = want or got
            assert all(torch.equal(a, b) for a, b in zip(got, want)), i


def test_attention_nodes_on_a_projection_give_rows(dev):
    """The nodes that take the fused projection [B, T, 3C] return [B, T, C]; the wrapper returns the heads [B, T, H, D] of the
    same values, and their gradients agree."""
    from oracle import attention as O
    from trainium_frontier_them_bones_amd import autograd as A, train_api as api
    B, T, H, D = 2, 128, 2, 64
    cos, sin = (t.to(dev) for t in O.rope_tables(T, D))
    qkv, gy = _t(dev, B, T, 3 * H * D, grad=True), _t(dev, B, T, H * D)
    y = A.RopeNormAttentionFn.apply(qkv, cos, sin, H, 0.125, api.RMS_EPS)
    z = api.nki_rope_attention(qkv, cos, sin, H, 0.125)
    assert y.shape == (B, T, H * D) and z.shape == (B, T, H, D) and torch.equal(y, z.reshape(B, T, H * D))
    (ga,), (gb,) = torch.autograd.grad(y, qkv, gy), torch.autograd.grad(z, qkv, gy.view(B, T, H, D))
    assert torch.equal(ga, gb)
    assert A.RopeAttentionFn.apply(qkv, cos, sin, H, 0.125).shape == (B, T, H * D)
