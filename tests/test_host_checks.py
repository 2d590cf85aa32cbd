"""The native host layer's checks of what a caller hands over, without a GPU: fake device tensors have shapes and types but no
memory, so a call that passes its checks ends where it asks for its first output ("No HIP GPUs") and reaches no kernel."""
import os

import pytest
import torch
from torch._subclasses.fake_tensor import FakeTensorMode

pytestmark = pytest.mark.filterwarnings("ignore:Accessing the data pointer of FakeTensor")
bf16, f32, u8 = torch.bfloat16, torch.float32, torch.uint8


@pytest.fixture
def A():
    from trainium_frontier_them_bones_amd import _lib, autograd
    if not os.path.exists(_lib.HOST_PATH):
        pytest.skip("host extension not built (run __graft_entry__.build())")
    if torch.cuda.is_available():
        pytest.skip("made for a machine without a GPU")
    with FakeTensorMode(allow_non_fake_inputs=True):
        yield autograd


def _t(*shape, dtype=bf16):
    return torch.empty(*shape, dtype=dtype, device="cuda")


def _passes(fn):
    """The call got through its checks."""
    with pytest.raises(RuntimeError, match="No HIP GPUs"):
        fn()


def _refused(fn, exc=ValueError):
    with pytest.raises(exc) as e:
        fn()
    assert "No HIP GPUs" not in str(e.value)


def _linear8_state(A, N, K, dw_fp8=False):
    st = A.Linear8State(dw_fp8=dw_fp8)
    st.sc, st.w8, st.w8t = _t(3, dtype=f32), _t(N, K, dtype=u8), _t(K, N, dtype=u8)
    return st


@pytest.mark.parametrize("res", [False, True])
@pytest.mark.parametrize("dw_fp8", [False, True])
def test_fp8_projection_refuses_other_operands(A, dw_fp8, res):
    """The rows come from x, its bytes may have any shape of as many; the bytes of the weight are the weight's."""
    w, st = _t(512, 256), _linear8_state(A, 512, 256, dw_fp8)
    x, r = _t(2, 128, 256), _t(2, 128, 512) if res else None
    call = A.Linear8Fn.apply
    _passes(lambda: call(x, w, st, 4.0, _t(256, 256, dtype=u8), r))
    _passes(lambda: call(x, w, st, 4.0, None, r))
    _passes(lambda: call(x, w, st, None, None, r))
    for x8 in (_t(384, 256, dtype=u8), _t(128, 256, dtype=u8), _t(256, 512, dtype=u8), _t(256, 128, dtype=u8)):
        _refused(lambda: call(x, w, st, 4.0, x8, r))
    _refused(lambda: call(x, w, st, 4.0, _t(256, 256), r), TypeError)
    for N, K in ((1024, 256), (256, 256), (512, 512), (512, 128)):
        _refused(lambda: call(x, w, _linear8_state(A, N, K, dw_fp8), 4.0, None, r))
    _refused(lambda: call(_t(2, 128, 512), w, st, 4.0, None, None))


def _mlp8_state(A, F, d, dw_fp8=False):
    st = A.Mlp8State(dw_fp8=dw_fp8)
    st.row, st.w8 = _t(16, dtype=f32), _t(4, F * d, dtype=u8)
    return st


@pytest.mark.parametrize("dw_fp8", [False, True])
def test_fp8_mlp_refuses_other_operands(A, dw_fp8):
    """The bytes are those of x itself (with bf16 weight gradients x is saved and contracted over the rows of the bytes), and
    the state's those of the call's weights."""
    d, F = 256, 512
    wf, wp, st = _t(F, d), _t(d, F), _mlp8_state(A, F, d, dw_fp8)
    call = A.Mlp8Fn.apply
    x, ragged = _t(2, 128, d), _t(3, 100, d)
    _passes(lambda: call(x, wf, wp, st))
    _passes(lambda: call(ragged, wf, wp, st))
    _passes(lambda: call(x, wf, wp, st, _t(256, d, dtype=u8), _t(2, 128, d)))
    for res in (None, _t(3, 100, d)):
        _refused(lambda: call(ragged, wf, wp, st, _t(384, d, dtype=u8), res))       # bytes of more rows than x has
        _refused(lambda: call(ragged, wf, wp, st, _t(300, d, dtype=u8), res))       # no whole tiles to read
    _refused(lambda: call(x, wf, wp, st, _t(128, d, dtype=u8)))
    _refused(lambda: call(x, wf, wp, st, _t(256, d)), TypeError)
    for F2, d2 in ((1024, d), (256, d), (F, 512)):
        _refused(lambda: call(x, wf, wp, _mlp8_state(A, F2, d2, dw_fp8)))
        _refused(lambda: call(_t(2, 128, d2), _t(F2, d2), _t(d2, F2), st))


def test_fp8_mlp_backward_refuses_rows_of_another_forward(A):
    """The backward rounds dy's rows up to whole tiles: r is compared with that count."""
    from trainium_frontier_them_bones_amd import ops
    d, F = 256, 512
    w8, row = _t(4, F * d, dtype=u8), _t(16, dtype=f32)
    for bwd in (lambda dy, r: ops.mlp8_bwd(dy, r, w8, row), lambda dy, r: ops.mlp8_bwd_q(dy, r, w8, row)):
        _passes(lambda: bwd(_t(256, d), _t(256, F)))
        _passes(lambda: bwd(_t(200, d), _t(256, F)))
        for rows, r in ((200, 200), (256, 128), (129, 128), (256, 384)):
            _refused(lambda: bwd(_t(rows, d), _t(r, F)))
        _refused(lambda: bwd(_t(256, d), _t(256, 1024)))
        _refused(lambda: bwd(_t(256, 512), _t(256, F)))
    _passes(lambda: ops.mlp_dw_proj(_t(256, d), _t(256, F)))
    _refused(lambda: ops.mlp_dw_proj(_t(256, d), _t(128, F)))


def test_block_head_with_a_skip_needs_its_gain(A):
    x, one = _t(4, 256), _t(1, dtype=f32)
    _passes(lambda: A.BlockHeadFn.apply(x, x, one, one, x, one, 1e-6))
    _refused(lambda: A.BlockHeadFn.apply(x, x, one, one, x, None, 1e-6), TypeError)


def test_an_empty_last_dimension_raises(A):
    """Rows are counted by the last dimension: an empty one is an error, not a division by zero that ends the process."""
    from trainium_frontier_them_bones_amd import ops
    from trainium_frontier_them_bones_amd import train_api as api
    e, one, tg = _t(4, 0), _t(1, dtype=f32), _t(4, dtype=torch.int64)
    b = _t(4, 0, dtype=u8)
    w, wt, w8 = _t(256, 0), _t(0, 256), _t(4, 0, dtype=u8)
    row, rows = _t(16, dtype=f32), _t(2, 16, dtype=f32)
    st, st8 = _mlp8_state(A, 256, 0), _linear8_state(A, 256, 0)
    for fn in (
            lambda: A.RMSNormFn.apply(e, None, 1e-6), lambda: A.RMSNormPassFn.apply(e, None, 1e-6, 4.0),
            lambda: A.AddRMSNormFn.apply(e, e, None, 1e-6), lambda: A.BlockHeadFn.apply(e, e, one, one, None, None, 1e-6),
            lambda: A.MixTailFn.apply(_t(1, 4, 0), one, 4), lambda: A.LinearFn.apply(e, w), lambda: A.LinearFn.apply(e, w, _t(4, 256)),
            lambda: A.Linear8Fn.apply(e, w, st8, 4.0), lambda: A.Mlp8Fn.apply(e, w, wt, st), lambda: A.NrMlpFn.apply(e, w, wt, st),
            lambda: A.MlpFusedFn.apply(e, w, wt), lambda: A.LmHeadLossFn.apply(e, w, tg, 0.0, "mean"),
            lambda: A.MoeMlp8Fn.apply(e, _t(2, 0, dtype=f32), _t(2, 256, 0), _t(2, 0, 256), None, 1, None),
            lambda: api.fused_loss(e, tg), lambda: api.fused_loss(e, tg, "none"), lambda: ops.matmul_res(e, wt, _t(4, 256)),
            lambda: ops.gemm_fp8(b, w8), lambda: ops.gemm_fp8_tn(b, b), lambda: ops.mlp8_backward_scales(e, row),
            lambda: ops.mlp8_fwd(e, w8, row, 256), lambda: ops.mlp8_bwd(e, _t(128, 256), w8, row), lambda: ops.mlp_dw_proj(e, _t(4, 256)),
            lambda: ops.mlp_bwd(e, _t(4, 256), w, wt), lambda: ops.lmhead_fwd(e, w, tg, 0.0)):
        _refused(fn)


def test_operands_of_the_same_rows_may_have_another_shape(A):
    """An operand that is added to x's rows or mixed into them has x's elements, in any shape; other counts are refused."""
    from trainium_frontier_them_bones_amd import train_api as api
    x, heads, more, less = _t(2, 128, 256), _t(2, 128, 4, 64), _t(3, 128, 256), _t(128, 256)
    one, w = _t(1, dtype=f32), _t(512, 256)
    wf, wp, st, st8 = _t(512, 256), _t(256, 512), _mlp8_state(A, 512, 256), _linear8_state(A, 512, 256)
    flat, wide = _t(256, 256), _t(256, 512)
    for fn in (lambda r: api.tail_norm2(x, r), lambda r: api.final_norm(x, r), lambda r: api.block_head(x, r, one, one),
               lambda r: api.head_skip(x, r, x, one, one, one), lambda r: api.head_skip(x, x, r, one, one, one),
               lambda r: A.Mlp8Fn.apply(x, wf, wp, st, None, r)):
        for r in (x, heads, flat, _t(2, 256, 128).transpose(1, 2)):
            _passes(lambda: fn(r))
        for r in (more, less, _t(1, 128, 256)):
            _refused(lambda: fn(r))
    for fn in (lambda r: A.LinearFn.apply(x, w, r), lambda r: A.Linear8Fn.apply(x, w, st8, 4.0, None, r)):
        _passes(lambda: fn(wide))
        _passes(lambda: fn(_t(2, 128, 8, 64)))
        _refused(lambda: fn(_t(128, 512)))
        _refused(lambda: fn(x))


def _node_calls(A):
    """class -> (all arguments, how many of them are needed)."""
    x, w, one = _t(2, 128, 256), _t(512, 256), _t(1, dtype=f32)
    qkv, cos = _t(2, 128, 768), _t(128, 32)
    q, wf, wp = _t(2, 4, 128, 64), _t(512, 256), _t(256, 512)
    st, st8, tg = _mlp8_state(A, 512, 256), _linear8_state(A, 512, 256), _t(256, dtype=torch.int64)
    gain, u, res, logits = _t(256), _t(2, 128, 256, dtype=u8), _t(2, 128, 512), _t(256, 512)
    router, ef, ep, bias = _t(4, 256, dtype=f32), _t(4, 512, 256), _t(4, 256, 512), _t(4, dtype=f32)
    return {
        A.RMSNormFn: ((x, gain, 1e-6), 3), A.RMSNormPassFn: ((x, gain, 1e-6, 4.0, False), 3), A.AddRMSNormFn: ((x, x, gain, 1e-6), 4),
        A.BlockHeadFn: ((x, x, one, one, x, one, 1e-6), 7), A.MixTailFn: ((x, one, 128), 3), A.Relu2Fn: ((x,), 1),
        A.LinearFn: ((x, w, res), 2), A.Linear8Fn: ((x, w, st8, 4.0, u, res), 4),
        A.CausalAttentionFn: ((q, q, q, 0.125, 0), 4), A.RopeAttentionFn: ((qkv, cos, cos, 4, 0.125), 5),
        A.RopeNormFn: ((_t(2, 128, 4, 64), cos, cos, 1e-6), 4), A.RopeNormAttentionFn: ((qkv, cos, cos, 4, 0.125, 1e-6, 0), 6),
        A.RopeNormAttentionHeadsFn: ((qkv, cos, cos, 4, 0.125, 1e-6, 0), 6), A.QkvRopeAttentionFn: ((x, _t(768, 256), cos, cos, 4, 0.125), 6), A.Mlp8Fn: ((x, wf, wp, st, u, x), 4),
        A.NrMlpFn: ((x, wf, wp, st, 1e-6), 4), A.MlpFusedFn: ((x, wf, wp), 3), A.LmHeadLossFn: ((x, w, tg, 15.0, "mean"), 5),
        A.FusedLossFn: ((logits, tg, 15.0), 3), A.ReducedLossFn: ((logits, tg, True, 15.0), 4), A.EmbeddingFn: ((tg, w), 2), A.MoeMlp8Fn: ((x, router, ef, ep, None, 2, bias, (0.1, 0.1), 8, {}), 7),
    }


def test_nodes_take_their_arguments_and_no_others(A):
    """A missing argument raises instead of standing for zero (a scale, an epsilon), one too many is not passed over."""
    may_be_none = ((A.Linear8Fn, 3), (A.LmHeadLossFn, 3), (A.FusedLossFn, 2), (A.ReducedLossFn, 3))   # a scale, a softcap
    for cls, (args, needed) in _node_calls(A).items():
        for n in range(needed, len(args) + 1):
            _passes(lambda: cls.apply(*args[:n]))
        _refused(lambda: cls.apply(*args[:needed - 1]), TypeError)
        _refused(lambda: cls.apply(*args, None), TypeError)
        for k, a in enumerate(args[:needed]):
            if isinstance(a, (float, A.Mlp8State, A.Linear8State)) and (cls, k) not in may_be_none:
                _refused(lambda: cls.apply(*args[:k], None, *args[k + 1:]), TypeError)
            if type(a) is int:
                _refused(lambda: cls.apply(*args[:k], None, *args[k + 1:]), TypeError)
    q = _t(2, 4, 128, 64)
    _passes(lambda: A.CausalAttentionFn.apply(q, q, q, 0.125, None))                        # no band
    _passes(lambda: A.LmHeadLossFn.apply(_t(256, 256), _t(512, 256), _t(256, dtype=torch.int64), None, "sum"))   # no softcap


def test_wrappers_for_sequences_take_three_dimensions(A):
    from trainium_frontier_them_bones_amd import train_api as api

    class Module:
        pass

    mlp = Module()
    mlp.c_fc, mlp.c_proj, mlp.tfb_mlp8 = Module(), Module(), _mlp8_state(A, 512, 256)
    mlp.c_fc.weight, mlp.c_proj.weight = _t(512, 256), _t(256, 512)
    for fn in (lambda x: api.mlp_fused8(mlp, x), lambda x: api.nr_mlp(mlp, x), lambda x: api.mlp_fused(mlp, x),
               lambda x: api.mix_tail(x, None, _t(1, dtype=f32))):
        _passes(lambda: fn(_t(2, 128, 256)))
        _refused(lambda: fn(_t(256, 256)))
        _refused(lambda: fn(_t(2, 2, 64, 256)))


def test_newton_schulz_stacks(A):
    from trainium_frontier_them_bones_amd import ops
    g, w = _t(2, 256, 128, dtype=f32), _t(3, 128, 256, dtype=f32)
    d, dw = _t(2, dtype=f32), _t(3, dtype=bf16)
    _passes(lambda: ops.ns5_stacks([(g, d)]))
    _passes(lambda: ops.ns5_stacks([(g, d), (w, dw)]))
    _refused(lambda: ops.ns5_stacks([]))
    _refused(lambda: ops.ns5_stacks([(g, d), (w, dw), (g, d)]))          # (the kernels take two)
    _refused(lambda: ops.ns5_stacks([(g, d), (_t(3, 128, 128, dtype=f32), dw)]))
    _refused(lambda: ops.ns5_stacks([(g, dw)]))
    far = torch.empty(3, 128, 256, dtype=f32, device="cuda:1")
    _refused(lambda: ops.ns5_stacks([(g, d), (far, dw)]))
    _refused(lambda: ops.ns5_stacks([(g, torch.empty(2, dtype=f32, device="cuda:1"))]))


@pytest.mark.parametrize("D", [64, 128])
def test_rotation_tables_of_the_projection(A, D):
    T, x, w = 256, _t(2, 256, 256), _t(3 * 256, 256)
    tab = lambda *s: (_t(*s), _t(*s))  # noqa: E731
    call = lambda c, s: (lambda: A.QkvRopeAttentionFn.apply(x, w, c, s, 256 // D, 0.1))  # noqa: E731
    _passes(call(*tab(T, D // 2)))
    _passes(call(*tab(2 * T, D // 2)))                    # (of a longer sequence)
    _refused(call(*tab(T, D // 4)))                       # of heads half as wide: the kernels would read past them
    _refused(call(*tab(T - 1, D // 2)))
    _refused(call(_t(T, D // 2), _t(T // 2, D // 2)))
