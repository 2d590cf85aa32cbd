"""The autograd nodes: the same role the reference's `*Fn` classes play (round1/source/train.py NkiAttnFn 8016, FcRelu2NNFn
4062, _ProjFn 3666, the loss head's LossHeadFn, Head2Fn 6599, _LinearGemm / _LmHeadDwSplit 8419-8711). `XFn.apply(...)` runs
the node of that name in the native host layer (csrc/host/nodes.cpp): forward and backward are C++ there, so that a small
call is not bound by the interpreter (a norm forward + backward on 256 rows: 58 us of host time as a Python autograd function).
Weight gradients follow the reference's in-place convention (round1/source/train.py:8463-8472): when a weight carries a
`grad_buf` tensor the gradient GEMM accumulates into it and autograd gets None for that weight; otherwise the gradient is
returned as usual. Nodes take any leading shape unless a class says otherwise.
"""
import math

import torch

from . import ops
from ._lib import native

bf16 = torch.bfloat16


class _Node:
    """Class attribute `apply`: the native function of the given name, looked up on first use (arguments are positional)."""

    def __init__(self, name):
        self.name = name

    def __get__(self, obj, cls):
        fn = getattr(native, self.name)
        cls.apply = staticmethod(fn)
        return fn


AMAX_HINT = "_tfb_amax_part"   # attribute on a gradient tensor: fp32 partials whose maximum is the tensor's amax
USE_AMAX_HINT = True           # False: consumers ignore the attribute and read the tensor for its amax


def _attach_amax(t, am):
    """Hang the amax partials of t's present contents on t, with t's version counter: an in-place update of t afterwards
    (autograd may add a second incoming gradient into it) makes the partials void."""
    native.attach_amax(t, am)
    return t


def _amax_hint(g, g2):
    """The amax partials the producer of gradient g attached to it, when g2 (the rows the caller will use) is g's own memory
    and g has not been written to since."""
    return native.amax_hint(g, g2) if USE_AMAX_HINT else None


class RMSNormFn:
    """(x, weight or None, eps): y = RMSNorm(x) * weight. A weight with a `dw_part` tensor has its gradient left there as
    partial sums, finished later with the other norms' by ops.norm_dw_finish."""
    apply = _Node("rmsnorm")


class RMSNormPassFn:
    """(x, weight, eps[, y8_scale[, bytes_only]]): (x, y[, y8]) = (x, RMSNorm(x) * weight[, e4m3(y * y8_scale)]) for a residual
    stream whose adds are made in the stores of the projections (LinearFn / Linear8Fn / Mlp8Fn with `res`): x is handed
    through so that the stream's gradient and the norm's meet in ONE backward launch (dx = g_x + J^T g_y), as in AddRMSNormFn.
    y8 is the operand cast of the fp8 GEMM that consumes y, made in the norm's pass (the norm prologue of
    round2/source/kernels/nki_mlp_nr8.py:1032 and nki_attn_nr8.py:929). bytes_only: the consumer reads y8 alone (Mlp8Fn with its
    weight gradients in fp8 too), so the bf16 rows of y are not written; the y handed back is a placeholder of y's shape without
    storage of its own (one NaN element, expanded), there only to carry the gradient edge. The gradient handed upstream carries
    its amax partials (AMAX_HINT): an fp8 MLP whose backward receives that very tensor takes its scales from them."""
    apply = _Node("rmsnorm_pass")


class AddRMSNormFn:
    """(x, res, weight, eps): (s, y) = (x + res, RMSNorm(x + res) * weight), the residual add fused in front of the norm
    (round1/source/train.py:6117 tail_norm2, 6826 final_norm)."""
    apply = _Node("add_rmsnorm")


class BlockHeadFn:
    """(x, x0, l1, l2, skip, l3, eps): (x_new, x_norm) = (l1 x + l2 x0 [+ l3 skip], RMSNorm(x_new)); gains are one-element
    tensors."""
    apply = _Node("block_head")


class LinearFn:
    """(x, w[, res]): y = x @ w^T with w [out, in] (nn.Linear layout), or bf16(res + bf16(x @ w^T)) with the residual add in the
    GEMM's store (nki_attn_nr8.py:1003); dW accumulates into w.grad_buf when present."""
    apply = _Node("linear")


class CausalAttentionFn:
    """(q, k, v, scale[, band]): nki_causal_attention: q, k, v [B, H, T, D] -> [B, T, H, D] (round1/source/train.py:8069).
    band = nw > 0: the reference's tile band (K/nki_attn_bandpro.py:1654): keys of the last nw 128-token tiles."""
    apply = _Node("attention")


class RopeAttentionFn:
    """(qkv, cos, sin, n_head, scale): attention straight from the fused projection output qkv [B, T, 3C]: RoPE of the q and k
    thirds into a buffer of its own (the input is left untouched), causal attention reading q, k from that buffer and v from qkv
    through strides, one dqkv [B, T, 3C] back (the call shape of nki_rope_attention, round1/source/train.py:8197, without its
    QK-norm)."""
    apply = _Node("rope_attention")


class RopeNormFn:
    """(x, cos, sin, eps): norm(apply_rotary_emb(x, cos, sin)) for x [B, T, H, D]: RoPE then the parameter-free per-head RMSNorm
    (round1/source/train.py:4411 RopeNormFn; rope_norm 4447 returns this transposed to [B, H, T, D])."""
    apply = _Node("rope_norm")


class RopeNormAttentionFn:
    """(qkv, cos, sin, n_head, scale, eps[, band]): nki_rope_attention (round1/source/train.py:8197, NkiRopeAttnFn 8135): causal
    SDPA(QKnorm(RoPE(q)), QKnorm(RoPE(k)), v) straight from the fused projection output qkv [B, T, 3C] -> [B, T, C], one dqkv
    [B, T, 3C] back. The input is not modified: the normalised q and k go to a fresh buffer, v is read in place through strides.
    band = nw > 0: the tile-band form (round2/source/train.py:4925 fused_rope_attention_band)."""
    apply = _Node("rope_norm_attention")


class RopeNormAttentionHeadsFn:
    """RopeNormAttentionFn with the result as [B, T, H, D], without a view node after it."""
    apply = _Node("rope_norm_attention_heads")


class QkvRopeAttentionFn:
    """(x, w_qkv, cos, sin, n_head, scale): the attention block's core in one node: qkv = rope(x @ w_qkv^T) (rotation in the
    projection's epilogue), causal attention on the thirds, and in backward the inverse rotation (head dimension 64: inside the
    attention kernels' stores; 128: a launch of its own) followed by the projection's dX and dW (accumulated into w_qkv.grad_buf
    when present). cos, sin [T, D / 2]."""
    apply = _Node("qkv_rope_attention")


class Linear8State:
    """Per-weight fp8 state of a projection, refreshed once per optimizer step: the weight's power-of-two scale
    (s, 1/s, amax on the device) and its e4m3 bytes in both layouts (forward_scales / precast_ref,
    round2/source/kernels/nki_attn_tt8g.py:700, 795)."""

    def __init__(self, limit=240.0, dw_fp8=False):
        self.limit = limit
        self.dw_fp8 = dw_fp8   # the weight gradient in fp8 too (attn8_weight_grad, round2/source/train.py:8232)
        self.sc = None
        self.w8 = self.w8t = None

    def refresh(self, w):
        self.sc = ops.amax_scale(w.detach(), self.limit, -24, 40)
        self.w8, self.w8t = ops.precast8(w.detach(), self.sc[0:1])


class Linear8Fn:
    """(x, w, state, x_scale[, x8[, res]]): y = x @ w^T with the forward in e4m3 x e4m3 and the input gradient in e5m2 x e4m3
    (per-tensor power-of-two scales, fp32 accumulation, one bf16 rounding); the weight gradient in bf16, or with state.dw_fp8 in
    fp8 from the gradient's e5m2 bytes and the forward's e4m3 activation bytes (round2/source/train.py:8232 attn8_weight_grad);
    either is accumulated into w.grad_buf when present. x_scale: the reference's constant (4 for an RMSNorm output) or None for
    the per-tensor amax scale of x. x8: the bytes e4m3(x * x_scale) when the norm that made x already cast them
    (RMSNormPassFn); res: a residual added in the GEMM's store (nki_attn_nr8.py:1003). The arithmetic of emulate_fwd /
    emulate_bwd (nki_attn_tt8g.py:745-757)."""
    apply = _Node("linear8")


class Mlp8State:
    """Per-layer fp8 state refreshed once per optimizer step: the scale row and the e4m3 weight pack
    (round2/source/train.py:6617 fp8_refresh_weights, 7003 mlp8_scales_into, 7267 mlp8_precast_into)."""

    def __init__(self, e4m3_limit=240.0, x_scale=4.0, dw_fp8=False):
        self.e4m3_limit, self.x_scale = e4m3_limit, x_scale
        self.dw_fp8 = dw_fp8   # weight gradients in fp8 too (round2/source/train.py:8209 under its switch 9k; R1 DW_ROWS)
        self.row = None
        self.w8 = None

    def refresh(self, w_fc, w_proj):
        self.row = ops.mlp8_forward_scales(w_fc.detach(), w_proj.detach(), self.e4m3_limit, self.x_scale)
        self.w8 = ops.mlp8_precast(w_fc.detach(), w_proj.detach(), self.row)


class Mlp8Fn:
    """(x, w_fc, w_proj, state[, x8[, res]]): y = c_proj(relu(c_fc(x))^2) with the four activation GEMMs in fp8 and the weight
    gradients in bf16 (K/nki_mlp_fused8.py:706 weight_grads) or, with state.dw_fp8, in fp8 from the bytes the other GEMMs
    multiplied (round2/source/train.py:8209 mlp8_weight_grads). x8: the bytes e4m3(x * state.x_scale) when the norm that made x
    already cast them (RMSNormPassFn); res: the block's residual, added in the second GEMM's store:
    y = bf16(res + bf16(MLP(x))) (nki_mlp_nr8.py:1032)."""
    apply = _Node("mlp8")


class NrMlpFn:
    """(x1, w_fc, w_proj, state[, eps]): x1 + MLP(rms_norm(x1)) for a dense block (round2/source/train.py:9168 NrMlp): the norm
    (parameter-free, eps 2^-23) also writes the MLP's e4m3 operand, the residual add is made in the second GEMM's store, and in
    the backward the norm's backward and the residual gradient's add are one launch (gx = g + J^T dxn)."""
    apply = _Node("nr_mlp")


LM_HEAD_ONE_PASS = True   # False: LmHeadLossFn always takes the GEMM with the lse epilogue and the separate loss backward


class LmHeadLossFn:
    """(x, W, targets, softcap, reduction): loss = reduce(CE(softcap(x @ W^T), targets)). When a gradient is wanted the forward is
    the plain LM-head GEMM followed by ONE pass over the logits that writes lse and the row losses and leaves, in place of the
    logits, their gradient for an upstream gradient of one; the backward is the two gradient GEMMs, each multiplying its product
    by the upstream scalar (a device value) before its rounding. The logits thus make one trip to HBM each way, and nothing
    recomputes an exponential. Without a gradient (or beyond the one-pass kernel's vocabulary limit) the GEMM with the
    log-sum-exp in its epilogue runs instead, and a backward from there writes dlogits in place of the logits first."""
    apply = _Node("lm_head_loss")


class FusedLossFn:
    """(logits, targets, softcap): the row losses [N] of materialised logits (round1/source/train.py:4691, reduction "none")."""
    apply = _Node("fused_loss")


class ReducedLossFn:
    """(logits, targets, mean, softcap): the reduced loss of materialised logits, the mean over the rows whose target counts or
    the sum (round1/source/train.py:4691): the reduction is a weight per row, made in one launch."""
    apply = _Node("reduced_loss")


class FusedLossMultiFn(torch.autograd.Function):
    """rows [N] = sum_k rw[k] (lse - (1 - eps) s_{t_k} - eps mean_v s_v) on materialised logits: several targets per row
    (round1/source/train.py:4870 LossMultiFn) and / or label smoothing (round2/source/train.py:6344 ChunkedLossHeadLS)."""

    @staticmethod
    def forward(ctx, logits2, tg, rw, softcap, eps):
        rows, lse = ops.loss_multi_fwd(logits2, tg, rw, softcap, eps)
        ctx.save_for_backward(logits2, tg, rw, lse)
        ctx.softcap, ctx.eps = softcap, eps
        return rows

    @staticmethod
    def backward(ctx, grows):
        logits2, tg, rw, lse = ctx.saved_tensors
        return ops.loss_multi_bwd(logits2, tg, rw, lse, grows.contiguous().float(), ctx.softcap, ctx.eps), None, None, None, None


class EmbeddingFn:
    """(idx, weight): weight rows gathered by idx; the gradient is accumulated into weight.grad_buf (fp32) when present."""
    apply = _Node("embedding")


class Relu2Fn:
    """(x): relu(x)^2 (round1/source/train.py:4161)."""
    apply = _Node("relu2")


def default_scale(D):
    return 1.0 / math.sqrt(D)


class Moe8State:
    """Per-layer fp8 state of the experts, refreshed once per optimizer step: a scale row and an e4m3 weight pack per
    expert (the reference's exp8_sc [E,128,16] / exp8_w8 buffers, round2/source/train.py:10900-10935)."""

    def __init__(self, e4m3_limit=240.0, x_scale=4.0, dw_fp8=False):
        """dw_fp8: the experts' weight gradients in fp8 as well, from the bytes the other four GEMMs multiplied (the
        reference's fp8 weight-gradient switch, round2/source/train.py:8209-8229, inside each expert's backward)."""
        self.e4m3_limit, self.x_scale, self.dw_fp8 = e4m3_limit, x_scale, dw_fp8
        self.rows = None
        self.w8 = None

    def refresh(self, w_fc, w_proj):
        E, F, d = w_fc.shape
        wf, wp = w_fc.detach(), w_proj.detach()
        if wf.is_contiguous() and wp.is_contiguous():      # the experts as E layers of one flat buffer: four launches
            self.rows, self.w8 = ops.mlp8_refresh_layers(wf[0], wp[0], F * d, E, self.e4m3_limit, self.x_scale)
            return
        rows = [ops.mlp8_forward_scales(wf[e], wp[e], self.e4m3_limit, self.x_scale) for e in range(E)]
        self.rows = torch.stack(rows).contiguous()
        self.w8 = torch.stack([ops.mlp8_precast(wf[e], wp[e], rows[e]) for e in range(E)]).contiguous()


class MoeMlp8Fn:
    """(h, router, w_fc, w_proj, state, topk, router_bias[, aux_weights[, capacity[, info]]]): the routed half of
    MoeMLP.forward_e8 (round2/source/train.py:11003-11067) with every expert on this GPU: router -> top-k -> dispatch -> grouped
    fp8 expert MLPs -> gated combine. h [.., d] bf16, router fp32 [E, d], w_fc [E, F, d], w_proj [E, d, F] bf16; router_bias fp32
    [E] or None (added to the logits).
    state None: the experts run in bf16 (MoeMLP.forward with moe_experts_local, round2/source/train.py:10941-11001, 10716: the
    kit's expression per expert, d and F multiples of 128).
    aux_weights = (alpha, beta): also returns (aux, stats) with aux = alpha lb + beta z, the router's weighted load-balance and z
    terms (round2/source/train.py:10779 moe_aux_terms; differentiable, its gradient joins the router's in the backward), and
    stats fp32 [2 + E] = (lb, z, the experts' load shares f_e). (alpha, beta, gamma) adds gamma times the per-sequence balance
    term (the reference's R2_MOE_AUX_SEQ, 10789-10792), the sequences being the rows of h [b, t, d].
    capacity: the reference's per-sequence count (round2/source/train.py:10555): each row of h [b, t, d] keeps its first
    `capacity` assignments per expert; None keeps everything.
    info: a dict that receives "kept" = the share of the assignments that hold a row (1 without a capacity), the first entry of
    the reference layer's statistics vector."""
    apply = _Node("moe")


class MlpFusedFn:
    """(x, w_fc, w_proj): the dense bf16 fused MLP y = c_proj(relu(c_fc(x))^2) with the fused kernels' rounding points; saves x
    and r only; dW accumulates into the weights' grad_buf when present (round2/source/kernels/nki_mlp_fused.py:408
    EmulatedFusedMlp; kernels :242, :290)."""
    apply = _Node("mlp_fused")


class MixTailFn:
    """(x, lam, T): (s1, xn2) = (x + lam shift1(x), RMSNorm(s1)) on a stream of sequences of T rows; gradients (gx, dlam)
    (round1/source/train.py:7330 MixTailFn)."""
    apply = _Node("mix_tail")
