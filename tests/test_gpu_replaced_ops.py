"""Functions of ops that a program replaces: the autograd nodes call what stands there, with the op's arguments, and its results
are what the node goes on with."""
import pytest
import torch

pytestmark = pytest.mark.gpu
bf16 = torch.bfloat16

# every op that some node calls
USED = """matmul matmul_res qkv_rope rmsnorm_fwd rmsnorm_fwd_q rmsnorm_bwd block_head_fwd block_head_bwd mix_tail_fwd mix_tail_bwd
amax_scale quant_fp8 gemm_fp8 gemm_fp8_res gemm_fp8_tn mlp8_backward_scales mlp8_fwd mlp8_bwd mlp8_bwd_q mlp8_dw8 mlp_dw_proj mlp_fwd
mlp_bwd relu2 relu2_bwd attn_fwd attn_bwd rope_ rope_norm_fwd rope_norm_bwd embedding_fwd embedding_bwd fill_f32_ loss_row_weights
loss_fwd loss_fwd_bwd loss_bwd lmhead_fwd moe_route moe_tables moe_gather moe_mlp8_fwd moe_mlp_fwd moe_combine moe_combine_bwd
moe_backward_scales_rowmax moe_mlp8_bwd moe_mlp8_bwd_q moe_quant_dout moe_mlp_bwd moe_dw8 moe_dw moe_aux_fwd moe_aux_seq_fwd
moe_route_bwd""".split()


def _nodes(dev):
    """Calls of every node, each with the tensors it is differentiated by."""
    from oracle import attention as O
    from trainium_frontier_them_bones_amd import autograd as A
    g = torch.Generator().manual_seed(7)

    def t(*shape, dtype=bf16, std=1.0, grad=True):
        return (std * torch.randn(*shape, generator=g)).to(dtype).to(dev).requires_grad_(grad)

    def state(cls, dw, *w):
        st = cls(dw_fp8=dw)
        st.refresh(*w)
        return st

    x, y, gain, one = t(2, 128, 256), t(2, 128, 256), t(256), [t(1, dtype=torch.float32) for _ in range(3)]
    odd = t(3, 100, 256)
    w, wq = t(256, 256, std=0.05), t(768, 256, std=0.05)
    wf, wp = t(512, 256, std=0.05), t(256, 512, std=0.05)
    router, ef, ep = t(4, 256, dtype=torch.float32, std=0.1), t(4, 512, 256, std=0.05), t(4, 256, 512, std=0.05)
    q, k, v = t(2, 4, 256, 64), t(2, 4, 256, 64), t(2, 4, 256, 64)
    qkv, qkv128, h4 = t(2, 256, 3 * 256), t(2, 256, 3 * 256), t(2, 256, 4, 64)
    c64, s64 = (a.to(dev) for a in O.rope_tables(256, 64))
    c128, s128 = (a.to(dev) for a in O.rope_tables(256, 128))
    xs = t(2, 256, 256)
    tg = torch.randint(0, 512, (2, 128), generator=g).to(dev)
    W, emb, logits = t(512, 256, std=0.05), t(512, 256), t(2, 128, 512)
    c64t, s64t = c64[:128].contiguous(), s64[:128].contiguous()
    calls = [
        (lambda: A.RMSNormFn.apply(x, gain, 1e-6), [x, gain]),
        (lambda: A.RMSNormPassFn.apply(x, gain, 1e-6)[1], [x, gain]),
        (lambda: A.RMSNormPassFn.apply(x, gain, 1e-6, 4.0)[1], [x, gain]),
        (lambda: A.AddRMSNormFn.apply(x, y, gain, 1e-6), [x, y, gain]),
        (lambda: A.BlockHeadFn.apply(x, y, one[0], one[1], x, one[2], 1e-6), [x, y] + one),
        (lambda: A.MixTailFn.apply(x, one[0], 128), [x, one[0]]),
        (lambda: A.Relu2Fn.apply(x), [x]),
        (lambda: A.LinearFn.apply(x, w), [x, w]),
        (lambda: A.LinearFn.apply(x, w, y), [x, w, y]),
        (lambda: A.CausalAttentionFn.apply(q, k, v, 0.125), [q, k, v]),
        (lambda: A.CausalAttentionFn.apply(q, k, v, 0.125, 1), [q, k, v]),
        (lambda: A.RopeAttentionFn.apply(qkv, c64, s64, 4, 0.125), [qkv]),
        (lambda: A.RopeAttentionFn.apply(qkv128, c128, s128, 2, 0.1), [qkv128]),
        (lambda: A.RopeNormFn.apply(h4, c64, s64, 1e-6), [h4]),
        (lambda: A.RopeNormAttentionFn.apply(qkv, c64, s64, 4, 0.125, 1e-6, 1), [qkv]),
        (lambda: A.RopeNormAttentionHeadsFn.apply(qkv128, c128, s128, 2, 0.1, 1e-6), [qkv128]),
        (lambda: A.QkvRopeAttentionFn.apply(x, wq, c64t, s64t, 4, 0.125), [x, wq]),
        (lambda: A.MlpFusedFn.apply(x, wf, wp), [x, wf, wp]),
        (lambda: A.LmHeadLossFn.apply(x, W, tg, 15.0, "mean"), [x, W]),
        (lambda: A.FusedLossFn.apply(logits, tg, 15.0), [logits]),
        (lambda: A.ReducedLossFn.apply(logits, tg, True, 15.0), [logits]),
        (lambda: A.EmbeddingFn.apply(tg, emb), [emb]),
    ]
    for dw in (False, True):
        st8, st, se = state(A.Linear8State, dw, w), state(A.Mlp8State, dw, wf, wp), state(A.Moe8State, dw, ef, ep)
        calls += [
            (lambda st8=st8: A.Linear8Fn.apply(x, w, st8, 4.0), [x, w]),
            (lambda st8=st8: A.Linear8Fn.apply(x, w, st8, None, None, y), [x, w, y]),
            (lambda st=st: A.Mlp8Fn.apply(odd, wf, wp, st), [odd, wf, wp]),
            (lambda st=st: A.Mlp8Fn.apply(x, wf, wp, st, None, y), [x, wf, wp, y]),
            (lambda st=st: A.NrMlpFn.apply(odd, wf, wp, st), [odd, wf, wp]),
            (lambda se=se: A.MoeMlp8Fn.apply(xs, router, ef, ep, se, 2, None, (0.1, 0.2)), [xs, router, ef, ep]),
            (lambda se=se: A.MoeMlp8Fn.apply(xs, router, ef, ep, se, 2, None, (0.1, 0.2, 0.3), 40, {}), [xs, router, ef, ep]),
        ]
    calls.append((lambda: A.MoeMlp8Fn.apply(xs, router, ef, ep, None, 1, None), [xs, router, ef, ep]))
    return calls


def _run(calls):
    out = []
    for call, wrt in calls:
        ys = call()
        ys = [ys] if torch.is_tensor(ys) else [a for a in ys if a.requires_grad]
        gs = [torch.ones_like(a) * 0.5 for a in ys]
        out += [a.detach() for a in ys] + list(torch.autograd.grad(ys, wrt, gs, allow_unused=True))
    return out


def _same(a, b):
    assert len(a) == len(b)
    for p, q in zip(a, b):
        assert (p is None) == (q is None) and (p is None or (p.shape == q.shape and p.dtype == q.dtype and torch.equal(p, q)))


def test_nodes_call_the_functions_that_replace_ops(dev, monkeypatch):
    """Each op in turn, and all together, behind a function that counts its calls and hands on to the op: it is called, and every
    output and gradient keeps its bits. The two-pass loss head is switched on for the ops that only it uses."""
    from trainium_frontier_them_bones_amd import _lib, autograd as A, ops
    calls = _nodes(dev)
    two_pass = [c for c in calls if len(c[1]) == 2 and c[1][1].shape == (512, 256) and c[1][1].requires_grad][:1]

    def everything():
        out = _run(calls)
        with monkeypatch.context() as m:
            m.setattr(A, "LM_HEAD_ONE_PASS", False)
            return out + _run(two_pass)

    want = everything()
    _same(everything(), want)
    seen = {}

    def counting(name, fn):
        def f(*a, **kw):
            seen[name] = seen.get(name, 0) + 1
            return fn(*a, **kw)
        return f

    for name in USED:
        print(name, flush=True)
        seen.clear()
        with monkeypatch.context() as m:
            m.setattr(ops, name, counting(name, getattr(ops, name)))
            assert list(_lib.REPLACED) == [name]
            _same(everything(), want)
        assert seen.get(name), name
        assert not _lib.REPLACED
    seen.clear()
    with monkeypatch.context() as m:
        for name in USED:
            m.setattr(ops, name, counting(name, getattr(ops, name)))
        _same(everything(), want)
    assert set(seen) == set(USED) - {"moe_quant_dout"}     # (its bytes come from moe_mlp8_bwd_q itself, which starts from dys)
    seen.clear()
    _same(everything(), want)
    assert not seen


def test_an_error_in_a_replacing_function_reaches_the_caller(dev, monkeypatch):
    from trainium_frontier_them_bones_amd import autograd as A, ops
    x = torch.randn(4, 64, device=dev).to(bf16).requires_grad_(True)

    def fail(*a):
        raise KeyError("mine")

    with monkeypatch.context() as m:
        m.setattr(ops, "rmsnorm_fwd", fail)
        with pytest.raises(KeyError, match="mine"):
            A.RMSNormFn.apply(x, None, 1e-6)
    y = A.RMSNormFn.apply(x, None, 1e-6)
    with monkeypatch.context() as m:
        m.setattr(ops, "rmsnorm_bwd", fail)
        with pytest.raises(KeyError, match="mine"):
            y.sum().backward()
