"""Attention behind the rotated projection with heads of 128: the node against the separate ones, with ops replaced, and in the model."""
import pytest
import torch

from helpers import rel_l2

pytestmark = pytest.mark.gpu
bf16 = torch.bfloat16


def _inputs(dev, B, T, H, Cin, D=128):
    from oracle import attention as O
    g = torch.Generator().manual_seed(B * T + H + Cin)
    x = torch.randn(B, T, Cin, generator=g).to(bf16).to(dev)
    w = (0.05 * torch.randn(3 * H * D, Cin, generator=g)).to(bf16).to(dev)
    go = torch.randn(B, T, H * D, generator=g).to(bf16).to(dev)
    return x, w, go, [t.to(dev) for t in O.rope_tables(T, D)]


def _separate(A, x, w, go, cos, sin, H):
    x, w = x.clone().requires_grad_(True), w.clone().requires_grad_(True)
    y = A.RopeAttentionFn.apply(A.LinearFn.apply(x, w), cos, sin, H, 0.09)
    y.backward(go)
    return y.detach(), x.grad, w.grad


# one tile of tokens; few tiles; ragged batches; a launch of the persistent kernel whose last 128 rows go by themselves
@pytest.mark.parametrize("B,T,H,Cin", [(1, 128, 1, 128), (2, 256, 2, 256), (3, 384, 4, 512), (5, 1920, 8, 1024)])
def test_node_equals_the_separate_nodes(dev, B, T, H, Cin):
    from trainium_frontier_them_bones_amd import autograd as A
    x, w, go, (cos, sin) = _inputs(dev, B, T, H, Cin)
    want = _separate(A, x, w, go, cos, sin, H)
    x1, w1 = x.clone().requires_grad_(True), w.clone().requires_grad_(True)
    y = A.QkvRopeAttentionFn.apply(x1, w1, cos, sin, H, 0.09)
    y.backward(go)
    for a, b in zip((y, x1.grad, w1.grad), want):
        assert torch.equal(a, b)
    # a token apart in memory, and the weight's gradient added to a buffer
    x2 = torch.cat([x, x], -1)[..., :Cin].requires_grad_(True)
    w2 = w.clone().requires_grad_(True)
    w2.grad_buf, w2.grad_fresh = torch.zeros_like(w), True
    A.QkvRopeAttentionFn.apply(x2, w2, cos, sin, H, 0.09).backward(go)
    assert torch.equal(x2.grad, want[1]) and torch.equal(w2.grad_buf, want[2]) and w2.grad is None


def test_replaced_ops_are_called_and_their_results_used(dev, monkeypatch):
    from trainium_frontier_them_bones_amd import autograd as A, ops
    B, T, H, Cin = 2, 256, 2, 256
    x, w, go, (cos, sin) = _inputs(dev, B, T, H, Cin)
    want = _separate(A, x, w, go, cos, sin, H)

    def node():
        x1, w1 = x.clone().requires_grad_(True), w.clone().requires_grad_(True)
        y = A.QkvRopeAttentionFn.apply(x1, w1, cos, sin, H, 0.09)
        y.backward(go)
        return y.detach(), x1.grad, w1.grad

    for name, times in (("matmul", 3), ("rope_", 2), ("attn_fwd", 1), ("attn_bwd", 1)):
        calls, own = [], getattr(ops, name)
        with monkeypatch.context() as m:
            m.setattr(ops, name, lambda *a, **kw: calls.append(1) or own(*a, **kw))
            assert all(torch.equal(a, b) for a, b in zip(node(), want)), name
        assert len(calls) == times, name
    with monkeypatch.context() as m:      # (an op of other paths: no call, the same results)
        m.setattr(ops, "relu2", lambda *a: 1 / 0)
        assert all(torch.equal(a, b) for a, b in zip(node(), want))
    own = ops.rope_
    with monkeypatch.context() as m:      # no rotation at all: plain attention on the projection
        m.setattr(ops, "rope_", lambda x, *a, **kw: x)
        got = node()
    plain = _separate(A, x, w, go, torch.ones_like(cos), torch.zeros_like(sin), H)
    assert own is ops.rope_ and all(torch.equal(a, b) for a, b in zip(got, plain))


@pytest.mark.parametrize("fuse", [True, False])
def test_model_with_heads_of_128(dev, fuse):
    """The attention half of every block against the oracle's on its own inputs (a bf16 path), and the losses of a few steps."""
    from oracle.model import OracleGPT
    from trainium_frontier_them_bones_amd.model import GPT, GPTConfig, zipf_tokens
    cfg = GPTConfig(n_layer=2, d_model=256, n_head=2, d_ff=1024, vocab=1024, seq_len=256, fuse_residual=fuse)
    m = GPT(cfg, dev, seed=1)
    o = OracleGPT(cfg, m.init_values)
    idx, tg = zipf_tokens(2, 256, cfg.vocab, seed=3)
    if fuse:
        m.trace = []
        m.zero_grad()
        m.backward(m.forward(idx.to(dev), tg.to(dev)))
        for i in range(cfg.n_layer):
            for t in o.p.values():
                t.grad = None
            t_in, t_out = m.trace[2 * i], m.trace[2 * i + 1]
            x_in = t_in.detach().cpu().clone().requires_grad_(True)
            x_out = o.attention_half(i, x_in)
            assert rel_l2(t_out, x_out) < 5e-3
            x_out.backward(t_out.grad.cpu())
            assert rel_l2(t_in.grad, x_in.grad) < 5e-3
            for n in ("norm1", "w_qkv", "w_o"):
                assert rel_l2(m.p["%s.%d" % (n, i)].grad_buf, o.p["%s.%d" % (n, i)].grad) < 5e-3, n
    m, o = GPT(cfg, dev, seed=1), OracleGPT(cfg, m.init_values)
    for _ in range(3):
        a, b = m.train_step(idx.to(dev), tg.to(dev)).item(), o.train_step(idx, tg).item()
        assert abs(a - b) < 1e-3 * b


@pytest.mark.parametrize("fuse", [True, False])
def test_head_dimensions_that_attention_refuses(dev, fuse):
    from trainium_frontier_them_bones_amd._lib import TfbError
    from trainium_frontier_them_bones_amd.model import GPT, GPTConfig, zipf_tokens
    idx, tg = (t.to(dev) for t in zipf_tokens(1, 128, 1024, seed=3))
    for heads in (8, 1):                  # 32 and 256
        m = GPT(GPTConfig(n_layer=1, d_model=256, n_head=heads, d_ff=1024, vocab=1024, seq_len=128, fuse_residual=fuse), dev)
        with pytest.raises(TfbError):
            m.forward(idx, tg)


def test_the_timed_entry_point_of_either_head_dimension(dev):
    """A program that times an entry point by its name gets its calls with the arguments that the header gives it."""
    from trainium_frontier_them_bones_amd import _lib, autograd as A, ops
    narrow, wide = [], []
    x, w, _, tabs = _inputs(dev, 1, 128, 4, 256, D=64)
    tabs128 = _inputs(dev, 1, 128, 2, 256)[3]
    _lib.TIMED.update(tfb_qkv_rope_fwd=narrow, tfb_qkv_rope_heads_fwd=wide)
    try:
        ops.qkv_rope(x[0], w, *tabs, 128, 512)
        A.QkvRopeAttentionFn.apply(x, w, *tabs, 4, 0.125)
        A.QkvRopeAttentionFn.apply(x, w, *tabs128, 2, 0.125)
    finally:
        del _lib.TIMED["tfb_qkv_rope_fwd"], _lib.TIMED["tfb_qkv_rope_heads_fwd"]
    torch.cuda.synchronize()
    assert [r[-1][5:10] for r in narrow] == [(128, 768, 256, 128, 512)] * 2 and [len(r[-1]) for r in narrow] == [11, 11]
    assert [r[-1][5:11] for r in wide] == [(128, 768, 256, 128, 512, 128)]
