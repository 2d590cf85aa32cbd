"""Functional layer over the C-ABI: torch tensors in, torch tensors out, one HIP launch (or a
short fixed sequence of launches) per call on torch's current stream. No autograd here (see
autograd.py) and no fallbacks: every function requires CUDA(ROCm) tensors and the built
library. torch supplies device memory and the stream; all arithmetic is in the HIP kernels.
"""
import sys
import types

import torch

from . import _lib
from ._lib import native

bf16 = torch.bfloat16


def _p(t):
    return None if t is None else t.data_ptr()


def _stream():
    return torch._C._cuda_getCurrentRawStream(torch._C._cuda_getDevice())


def _chk(t, dtype=bf16):
    if t is None:
        return
    if not t.is_cuda:
        raise RuntimeError("tfb ops need device tensors (the HIP kernels are the only implementation)")
    if t.dtype != dtype:
        raise TypeError("expected %s, got %s" % (dtype, t.dtype))
    if not t.is_contiguous():
        raise RuntimeError("tensor must be contiguous")


# ------------------------------------------------------------------------------------------ GEMM
def matmul(a, b, trans_a=False, trans_b=False, out=None, accumulate=False, out_dtype=bf16, alpha=None):
    """op(a) @ op(b) with fp32 accumulation. a is [M,K] (or [K,M] with trans_a), b is [K,N] (or [N,K] with
    trans_b). `out` (bf16 or fp32) may be given; accumulate=True adds into it (one rounding). alpha: a 1-element fp32
    device tensor the product is multiplied by before that rounding (no host read-back)."""
    if alpha is None:
        return native.tfb_gemm_bf16(a, b, trans_a, trans_b, out, accumulate, out_dtype == torch.float32)
    return native.tfb_gemm_bf16_scaled(a, b, trans_a, trans_b, out, accumulate, out_dtype == torch.float32, alpha)


def matmul_res(a, b, res, trans_b=False):
    """bf16(res + bf16(a @ op(b))): a projection with the residual add that follows it made in the GEMM's store (equal to
    matmul followed by a bf16 add, bit for bit). a [M,K]; b [K,N] or, with trans_b, [N,K]; res [M,N]."""
    return native.tfb_gemm_bf16_res(a, b, res, trans_b)


def qkv_rope(x2, w, cos, sin, T, rot_cols):
    """rope(x2 @ w^T): the fused attention projection [M, N] with the rotary embedding of its first rot_cols columns
    (heads of 64) applied in the GEMM epilogue; row m is token m % T."""
    return native.tfb_qkv_rope_fwd(x2, w, cos, sin, T, rot_cols)


# ------------------------------------------------------------------------------------------ norms
def rmsnorm_fwd(x, weight=None, eps=2.0 ** -23, res=None):
    """y = RMSNorm(s) * weight with s = x (res None) or bf16(x + res). Returns (s, y, inv[rows] fp32)."""
    return native.tfb_rmsnorm_fwd(x, weight, eps, res)


def rmsnorm_fwd_q(x, weight=None, eps=2.0 ** -23, res=None, y8_scale=4.0, want_y=True, rows_out=0):
    """rmsnorm_fwd that also returns y8 = e4m3(bf16(y) * y8_scale) bytes, the operand cast of the fp8 GEMM that consumes y
    (equal to quant_fp8(y, y8_scale), bit for bit). Returns (s, y, inv, y8); want_y False: the bf16 rows are not written and
    y is None (for a consumer that reads only the bytes). rows_out: y and y8 get that many rows, those beyond x's zero."""
    if rows_out:
        return native.tfb_rmsnorm_fwd_q_pad(x, weight, eps, res, y8_scale, want_y, rows_out)
    return native.tfb_rmsnorm_fwd_q(x, weight, eps, res, y8_scale, want_y)


def rmsnorm_bwd(gy, s, inv, weight=None, gs=None, dw=None, accumulate=False, part=None, want_amax=False):
    """dx = gs + J^T(gy) for y = RMSNorm(s) * weight. Returns (dx, dw fp32 [C] or None); a given dw is written, or
    added into with accumulate=True. With `part` (fp32 [tfb_norm_bwd_blocks(rows), C]) the weight gradient is left there
    as partial sums for norm_dw_finish and None is returned for it. want_amax: a third value, fp32 [tfb_norm_bwd_blocks(rows)]
    whose maximum is amax(dx) (per-workgroup partials, for mlp8_backward_scales(..., amax_part=))."""
    if want_amax:
        return native.tfb_rmsnorm_bwd_amax(gy, s, inv, weight, gs, dw, accumulate, part, True)
    return native.tfb_rmsnorm_bwd(gy, s, inv, weight, gs, dw, accumulate, part, False)


def norm_bwd_blocks(rows):
    return int(_lib.lib().tfb_norm_bwd_blocks(rows))


def norm_dw_finish(parts, dw, rows, accumulate=False):
    """dw [count, C] fp32 (+)= the weight gradients whose partial sums rmsnorm_bwd(part=parts[i]) left in parts
    [count, blocks, C]: one launch for all of them."""
    _chk(parts, torch.float32), _chk(dw, torch.float32)
    count, nb, C = parts.shape
    if tuple(dw.shape) != (count, C) or nb != norm_bwd_blocks(rows):
        raise ValueError("parts [count, blocks, C], dw [count, C]")
    _lib.call("tfb_norm_dw_finish", _p(parts), _p(dw), count, nb * C, C, int(accumulate), rows, C, _stream())
    return dw


def block_head_fwd(x, x0, gains, skip=None, eps=2.0 ** -23):
    """x_new = l1*x + l2*x0 (+ l3*skip), x_norm = RMSNorm(x_new). gains: fp32 device tensor [3]."""
    return native.tfb_block_head_fwd(x, x0, gains, skip, eps)


def block_head_bwd(g_new, g_norm, x, x0, x_new, inv, gains, skip=None):
    """Returns (dx, dx0, dskip or None, dgains fp32 [4] = sum G.x, G.x0, G.skip, 0)."""
    return native.tfb_block_head_bwd(g_new, g_norm, x, x0, x_new, inv, gains, skip)


# ------------------------------------------------------------------------------------------ fp8 MLP
NSC = 16
FMT_E4M3, FMT_E5M2 = 0, 1
fp8_dtypes = (torch.float8_e4m3fn, torch.float8_e5m2)


def _scratch(device, nfloats):
    return torch.empty(nfloats, dtype=torch.float32, device=device)


def _scale_arg(x_scale):
    """(float, device pointer) for an activation scale given as a python float or as a 1-element fp32 device tensor."""
    if isinstance(x_scale, torch.Tensor):
        _chk(x_scale, torch.float32)
        if x_scale.numel() != 1:
            raise ValueError("a device activation scale is one fp32 element")
        return 0.0, _p(x_scale)
    return float(x_scale), None


def mlp8_forward_scales(w_fc, w_proj, e4m3_limit=240.0, x_scale=4.0):
    """The layer's fp32 [16] scale row, computed on the device from the bf16 weights (w_fc [F,d], w_proj [d,F]).
    x_scale: python float (the reference's constant 4) or a 1-element fp32 device tensor (no host synchronisation)."""
    _chk(w_fc), _chk(w_proj)
    F, d = w_fc.shape
    if tuple(w_proj.shape) != (d, F):
        raise ValueError("w_proj must be [d, F]")
    row = torch.empty(NSC, dtype=torch.float32, device=w_fc.device)
    scr = _scratch(w_fc.device, _lib.lib().tfb_mlp8_scale_scratch_floats(F))
    xf, xd = _scale_arg(x_scale)
    _lib.call("tfb_mlp8_forward_scales", _p(w_fc), _p(w_proj), _p(row), _p(scr), F, d, float(e4m3_limit), xf, xd, _stream())
    return row


def mlp8_refresh_layers(w_fc0, w_proj0, layer_stride, layers, e4m3_limit=240.0, x_scale=4.0, rows=None, w8=None):
    """Scale rows [layers, 16] and e4m3 packs [layers, 4, F*d] of `layers` MLPs whose weights share one flat buffer:
    layer i's w_fc [F, d] starts layer_stride elements after layer i-1's (w_fc0, w_proj0: layer 0's), likewise w_proj.
    Six launches whatever the layer count; rows / w8 may be given to be overwritten."""
    _chk(w_fc0), _chk(w_proj0)
    F, d = w_fc0.shape
    if tuple(w_proj0.shape) != (d, F):
        raise ValueError("w_proj must be [d, F]")
    dev = w_fc0.device
    if rows is None:
        rows = torch.empty(layers, NSC, dtype=torch.float32, device=dev)
    if w8 is None:
        w8 = torch.empty(layers, 4, F * d, dtype=torch.uint8, device=dev)
    _chk(rows, torch.float32), _chk(w8, torch.uint8)
    scr = _scratch(dev, layers * _lib.lib().tfb_mlp8_scale_scratch_floats(F))
    _lib.call("tfb_mlp8_refresh_layers", _p(w_fc0), _p(w_proj0), int(layer_stride), int(layers), _p(rows), _p(w8), _p(scr),
              F, d, float(e4m3_limit), float(x_scale), _stream())
    return rows, w8


def mlp8_backward_scales(dy2, row, amax_part=None):
    """The backward call's scale row from amax(dy2), or from amax_part (fp32 partials whose maximum is that amax, as
    rmsnorm_bwd(want_amax=True) leaves them for the dx it wrote) without reading dy2."""
    if amax_part is not None:
        return native.tfb_mlp8_backward_scales_part(dy2, row, amax_part)
    return native.tfb_mlp8_backward_scales(dy2, row)


def amax_scale(x, limit, e_lo, e_hi):
    """fp32 [3] = (s, 1/s, amax): s the largest power of two in [2^e_lo, 2^e_hi] with amax(x) * s <= limit."""
    return native.tfb_amax_scale(x, limit, e_lo, e_hi)


def quant_fp8(x, scale, fmt=FMT_E4M3):
    """uint8-carried fp8 of x * scale; scale a python float or a 1-element fp32 device tensor (no host sync)."""
    return native.tfb_quant_fp8(x, scale, fmt)


def precast8(w, scale):
    """(w8 [R,C], w8T [C,R]) uint8: e4m3(w * scale) in both byte layouts; scale a 1-element fp32 device tensor."""
    _chk(w), _chk(scale, torch.float32)
    R, C = w.shape
    w8 = torch.empty(R, C, dtype=torch.uint8, device=w.device)
    w8t = torch.empty(C, R, dtype=torch.uint8, device=w.device)
    _lib.call("tfb_precast8", _p(w), _p(scale), _p(w8), _p(w8t), R, C, _stream())
    return w8, w8t


def gemm_fp8(a8, b8, fmt_a=FMT_E4M3, dq_a=None, dq_b=None, dq=1.0):
    """bf16 [M,N] = (a8 [M,K] @ b8 [N,K]^T) * dq * dq_a * dq_b; a8 e4m3 or e5m2 bytes, b8 e4m3 bytes; dq_a, dq_b
    1-element fp32 device tensors (or None)."""
    return native.tfb_gemm_fp8(a8, b8, fmt_a, dq_a, dq_b, dq)


def gemm_fp8_res(a8, b8, res, dq_a=None, dq_b=None, dq=1.0):
    """bf16(res + bf16((a8 [M,K] @ b8 [N,K]^T) * dq * dq_a * dq_b)): gemm_fp8 (e4m3 activations) with the residual add
    in the store, equal to gemm_fp8 followed by a bf16 add bit for bit."""
    return native.tfb_gemm_fp8_res(a8, b8, FMT_E4M3, dq_a, dq_b, dq, res)


def gemm_fp8_tn(g8, a8, fmt_g=FMT_E5M2, fmt_a=FMT_E4M3, s_g=None, s_a=None, imm=1.0, out=None, accumulate=False,
                out_dtype=bf16):
    """[O,D] (+)= (g8 [M,O]^T @ a8 [M,D]) * imm / (s_g s_a): a weight gradient in fp8 (dw8_grad,
    round2/source/train.py:8185). s_g, s_a: 1-element fp32 device tensors (the scales the bytes were cast at) or None."""
    return native.tfb_gemm_fp8_tn(g8, a8, fmt_g, fmt_a, s_g, s_a, imm, out, accumulate, out_dtype == torch.float32)


def mlp8_precast(w_fc, w_proj, row):
    """uint8 [4, F*d]: w_fc and w_proj cast once to e4m3 at the row's scales, each in both byte layouts."""
    _chk(w_fc), _chk(w_proj), _chk(row, torch.float32)
    F, d = w_fc.shape
    w8 = torch.empty(4, F * d, dtype=torch.uint8, device=w_fc.device)
    _lib.call("tfb_mlp8_precast", _p(w_fc), _p(w_proj), _p(row), _p(w8), F, d, _stream())
    return w8


def mlp8_fwd(x2, w8, row, F, x_scale=4.0, want_x8=False, x8=None, res=None):
    """y [M,d], r [M,F] (bf16): the fp8 forward. x_scale: python float (the reference's constant 4) or a device scalar.
    want_x8 also returns x8 = e4m3(x x_scale) [M,d] bytes (the fp8 weight gradient's operand). A given x8 (from
    rmsnorm_fwd_q) is used instead of casting x2; with res [M,d], y = bf16(res + bf16(MLP(x))) (the block's residual add
    made in the second GEMM's store)."""
    if res is None:
        y, r, x8 = native.tfb_mlp8_fwd(x2, w8, row, F, x_scale, x8)
    else:
        y, r, x8 = native.tfb_mlp8_fwd_res(x2, w8, row, F, x_scale, x8, res)
    return (y, r, x8) if want_x8 else (y, r)


def mlp8_bwd(dy2, r, w8, row, want_h=True):
    """dx [M,d], h [M,F] (or None), dpre [M,F]: the fp8 backward; row = this call's backward row."""
    return native.tfb_mlp8_bwd(dy2, r, w8, row, want_h)


def mlp8_bwd_q(dy2, r, w8, row, e4m3_limit=240.0, want_dpre=True):
    """The fp8 backward keeping the byte tensors of the fp8 weight gradients: (dx [M,d], dpre [M,F] (None without
    want_dpre: the fp8 weight gradients read only its bytes), dp8 [M,F] e5m2 bytes, hq8 [M,F] = e4m3(min(bf16(r^2) s_h,
    e4m3_limit)) bytes, dy8 [M,d] e5m2 bytes)."""
    return native.tfb_mlp8_bwd_q(dy2, r, w8, row, e4m3_limit, want_dpre)


def mlp8_dw8(x8, dp8, hq8, dy8, row, x_scale=4.0, dw_fc=None, dw_proj=None, accumulate=False, out_dtype=bf16):
    """(dw_fc [F,d], dw_proj [d,F]) (+)= the fp8 weight gradients from the forward's x8 and the backward's dp8, hq8, dy8
    (mlp8_weight_grads under the fp8 weight-gradient switch, round2/source/train.py:8209)."""
    return native.tfb_mlp8_dw8(x8, dp8, hq8, dy8, row, x_scale, dw_fc, dw_proj, accumulate, out_dtype == torch.float32)


def mlp_dw_proj(dy2, r, out=None, accumulate=False, out_dtype=bf16):
    """dw_proj [d,F] (+)= dy^T @ bf16(r^2) without materialising h."""
    return native.tfb_mlp_dw_proj(dy2, r, out, accumulate, out_dtype == torch.float32)


# ------------------------------------------------------------------------------------------ attention
import ctypes as _ct

_L3 = _ct.c_long * 3


def _bht(t, layout):
    """(batch, head, token) element strides of a 4-D tensor given as "bhtd" or "bthd", for a call of the C-ABI itself."""
    if layout == "bhtd":
        return _L3(t.stride(0), t.stride(1), t.stride(2))
    return _L3(t.stride(0), t.stride(2), t.stride(1))


def attn_fwd(q, k, v, scale, layout="bhtd", band=0):
    """q, k, v: 4-D views [B,H,T,D] ("bhtd") or [B,T,H,D] ("bthd"), arbitrary batch/head/token strides.
    Returns o [B,T,H,D] contiguous and lse [B,H,T] fp32. band = nw > 0: the reference's tile band (a query of 128-token
    tile i sees the keys k <= q of tiles i - nw + 1 .. i; K/nki_attn_bandpro.py:1654); 0: all keys k <= q."""
    if band:
        return native.tfb_attn_fwd_band(q, k, v, scale, layout, band)
    return native.tfb_attn_fwd(q, k, v, scale, layout)


def attn_bwd(q, k, v, o, do, lse, scale, layout="bhtd", dq=None, dk=None, dv=None, out_layout="bhtd", rope=None, band=0):
    """Gradients of attn_fwd. o, do are [B,T,H,D]. dq/dk/dv may be given as (strided) views with `out_layout`;
    otherwise dq, dk are allocated [B,H,T,D] and dv [B,T,H,D] (returned as a [B,H,T,D] view), as the reference returns.
    rope = (cos, sin) (bf16 [T, D/2]): dq and dk come back with the inverse rotation applied (D = 64)."""
    if dq is None:
        if q.dim() != 4:
            raise ValueError("attention tensors are 4-D")
        B, H, T, D = q.shape if layout == "bhtd" else (q.shape[0], q.shape[2], q.shape[1], q.shape[3])
        dq = torch.empty(B, H, T, D, dtype=bf16, device=q.device)
        dk = torch.empty(B, H, T, D, dtype=bf16, device=q.device)
        dv = torch.empty(B, T, H, D, dtype=bf16, device=q.device).permute(0, 2, 1, 3)
        out_layout = "bhtd"
    args = (q, k, v, o, do, lse, scale, layout, dq, dk, dv, out_layout)
    if band:
        native.tfb_attn_bwd_band(*args, *(rope or (None, None)), band)
    elif rope is not None:
        native.tfb_attn_bwd_rope(*args, *rope)
    else:
        native.tfb_attn_bwd(*args)
    return dq, dk, dv


def attn_bwd_static_max_rows():
    """The largest B * H * T attn_bwd_static takes (the size of the library's static scratch array)."""
    return int(_lib.lib().tfb_attn_bwd_static_max_rows())


def attn_bwd_static(q, k, v, o, do, lse, scale, dq, dk, dv, layout="bhtd", out_layout="bhtd"):
    """attn_bwd into caller-provided dq, dk, dv through the entry point that allocates nothing: its row-statistic scratch
    is a static device array inside the library (B * H * T <= tfb_attn_bwd_static_max_rows(); TfbError status 4 beyond).
    Calls that overlap on one GPU share that array and race; this wrapper creates no tensor either. The FIRST call on a
    device looks up the array's address: make one call eagerly before capturing this one into a HIP graph."""
    native.tfb_attn_bwd_static(q, k, v, o, do, lse, scale, layout, dq, dk, dv, out_layout)
    return dq, dk, dv


# ------------------------------------------------------------------------------------------ elementwise
def relu2(x):
    return native.tfb_relu2(x, None, 0)


def relu2_bwd(x, gy):
    return native.tfb_relu2(x, gy, 1)


def relu2_bwd_from_h(h, dh):
    return native.tfb_relu2(h, dh, 2)


def rope_(x, cos, sin, T, nheads, D, inverse=False, out=None):
    """Rotate the first nheads*D columns of each row of x ([rows, row_stride] view, contiguous rows) in place
    (or into `out`). cos, sin: bf16 [T, D/2]; row r is token r % T."""
    native.tfb_rope(x, cos, sin, T, nheads, D, inverse, out)
    return x if out is None else out


def rope_norm_fwd(x, cos, sin, T, nheads, D, eps=2.0 ** -23, want_r=True):
    """RoPE then parameter-free RMSNorm of each of the first `nheads` heads (D columns each) of every row of x
    ([rows, row_stride] view). Returns (y [rows, nheads*D] normalised, r [rows, nheads*D] rotated or None,
    inv [rows, nheads] fp32)."""
    return native.tfb_rope_norm_fwd(x, cos, sin, T, nheads, D, eps, want_r)


def rope_norm_bwd(g, r, inv, cos, sin, T, nheads, D, out=None):
    """The gradient of rope_norm_fwd's input from g (gradient of y; [rows, row_stride] view), the saved r and inv; written
    into `out` ([rows, row_stride] view) or a fresh [rows, nheads*D] tensor."""
    return native.tfb_rope_norm_bwd(g, r, inv, cos, sin, T, nheads, D, out)


def resmix_bwd(g, x, x0, ab):
    """dx = g*a, dx0 = g*b, dab = (sum g*x, sum g*x0) for x_new = a*x + b*x0; ab: fp32 device [2]."""
    _chk(g), _chk(x), _chk(x0), _chk(ab, torch.float32)
    dx, dx0 = torch.empty_like(g), torch.empty_like(g)
    nb = _lib.lib().tfb_resmix_bwd_blocks(g.numel())
    part = torch.empty(2 * nb, dtype=torch.float32, device=g.device)
    dab = torch.empty(2, dtype=torch.float32, device=g.device)
    _lib.call("tfb_resmix_bwd", _p(g), _p(x), _p(x0), _p(ab), _p(dx), _p(dx0), _p(part), _p(dab), g.numel(), _stream())
    return dx, dx0, dab


def embedding_fwd(idx, weight):
    """weight rows gathered by idx; an id outside [0, V) gives a zero row (and receives no gradient in embedding_bwd)."""
    return native.tfb_embedding_fwd(idx, weight)


def embedding_bwd(idx, dy, dw, grouped=True):
    """dw (fp32 [V, C]) += scatter of dy rows by idx. grouped: rows sorted by token on the device and summed per token
    (deterministic order inside a token's run); False: one fp32 atomic add per element (the plain entry point)."""
    if grouped:
        native.tfb_embedding_bwd_grouped(idx, dy, dw)
        return dw
    _chk(dy), _chk(dw, torch.float32)
    idx = idx.contiguous()
    _lib.call("tfb_embedding_bwd", _p(idx), int(idx.dtype == torch.int64), _p(dy), _p(dw), idx.numel(), dy.shape[-1], dw.shape[0],
              _stream())
    return dw


def fill_f32_(t, val=0.0):
    native.tfb_fill_f32(t, val)
    return t


def adamw_(p, g, m, v, step, lr, beta1, beta2, eps, weight_decay, p_bf16=None):
    """One in-place AdamW update of the fp32 master p (and its optional bf16 copy) from g (fp32 or bf16)."""
    native.tfb_adamw(p, g, m, v, step, lr, beta1, beta2, eps, weight_decay, p_bf16)


# ------------------------------------------------------------------------------------------ loss head
def _tg(targets):
    if targets.dtype not in (torch.int64, torch.int32) or not targets.is_cuda:
        raise TypeError("targets must be an int32/int64 device tensor")
    return targets.contiguous()


def loss_fwd(logits2, targets, softcap=15.0, row_w=None):
    """Row losses (already multiplied by row_w) and lse, from bf16 logits [N, V]; targets < 0 are ignored."""
    return native.tfb_loss_fwd(logits2, targets, row_w, softcap)


def loss_bwd(logits2, targets, lse, grow, softcap=15.0, inplace=False):
    """dlogits bf16 [N, V]; grow fp32 [N] = d(total)/d(row loss) * row weight."""
    return native.tfb_loss_bwd(logits2, targets, lse, grow, softcap, inplace)


def loss_row_weights(targets, reduction="mean", V=None):
    """fp32 [N] weights of the row losses in the reduced loss: valid / max(1, count of valid) for "mean", valid for "sum";
    a row is valid when 0 <= t < V (the rows the loss kernels give a loss to; V None: when t >= 0)."""
    return native.tfb_loss_row_weights(targets, reduction == "mean", V)


LOSS_FWD_BWD_MAX_V = 65536


def loss_fwd_bwd(logits2, targets, row_w=None, softcap=15.0):
    """(loss rows fp32 [N], lse fp32 [N]) as loss_fwd gives them, and logits2 OVERWRITTEN by the gradient of sum(rows):
    row_w (softmax - onehot) (1 - tanh^2), what loss_bwd gives for grow = row_w. One pass over the logits; V <= 65536."""
    return native.tfb_loss_fwd_bwd(logits2, targets, row_w, softcap)


def loss_multi_fwd(logits2, targets, row_w, softcap=15.0, eps=0.0):
    """Row losses sum_k row_w[k] (lse - (1 - eps) s_{t_k} - eps mean_v s_v) and lse; targets [K, N] (int64 / int32, < 0 =
    weight 0), row_w fp32 [K, N]."""
    _chk(logits2), _chk(row_w, torch.float32)
    tg = _tg(targets)
    K, N = tg.shape
    V = logits2.shape[1]
    if tuple(row_w.shape) != (K, N) or logits2.shape[0] != N:
        raise ValueError("targets [K, N], row_w [K, N], logits [N, V]")
    loss = torch.empty(N, dtype=torch.float32, device=logits2.device)
    lse = torch.empty(N, dtype=torch.float32, device=logits2.device)
    _lib.call("tfb_loss_multi_fwd", _p(logits2), _p(tg), int(tg.dtype == torch.int64), _p(row_w), K, float(eps), _p(loss),
              _p(lse), N, V, float(softcap or 0.0), _stream())
    return loss, lse


def loss_multi_bwd(logits2, targets, row_w, lse, g, softcap=15.0, eps=0.0, inplace=False):
    """dlogits bf16 [N, V] of loss_multi_fwd; g fp32 [N] = d(total)/d(row loss)."""
    _chk(logits2), _chk(row_w, torch.float32), _chk(lse, torch.float32), _chk(g, torch.float32)
    tg = _tg(targets)
    K, N = tg.shape
    V = logits2.shape[1]
    out = logits2 if inplace else torch.empty_like(logits2)
    _lib.call("tfb_loss_multi_bwd", _p(logits2), _p(tg), int(tg.dtype == torch.int64), _p(row_w), K, float(eps), _p(lse),
              _p(g), _p(out), N, V, float(softcap or 0.0), _stream())
    return out


def lmhead_fwd(x2, W, targets, softcap=None, row_w=None):
    """logits = x2 @ W^T (W [V, d]) with the row log-sum-exp fused into the GEMM epilogue.
    Returns (logits bf16 [N, V], loss rows fp32 [N], lse fp32 [N])."""
    return native.tfb_lmhead_fwd(x2, W, targets, softcap, row_w)


# ------------------------------------------------------------------------------------------ mixture of experts
def moe_max_rows(N, E, topk):
    return _lib.lib().tfb_moe_max_rows(N, E, topk)


def moe_route(h2, wr, topk, bias=None, want_logits=False):
    """(p fp32 [N,E], idx int32 [N,topk], gate fp32 [N,topk], logits or None) from h2 bf16 [N,d], wr fp32 [E,d]."""
    return native.tfb_moe_route(h2, wr, topk, bias, want_logits)


def moe_tables(idx, E, seq_len=None, capacity=None):
    """Slot tables for the ragged layout: dict(cnt, seg, tile_expert, slot, tok, ksel, rmax). Dropless by default; with
    seq_len and capacity the reference's per-sequence capacity (round2/source/train.py:10555-10634): each sequence keeps its
    first `capacity` assignments per expert, the rest get slot -1; the dict then also holds cnt_all (every assignment)."""
    if capacity is None:
        return native.tfb_moe_tables(idx, E)
    return native.tfb_moe_tables_cap(idx, E, seq_len, capacity)


def moe_gather(h2, tab, x_scale=4.0, want_xs=True):
    """(xs bf16 [rmax,d], xs8 uint8 [rmax,d]); x_scale None: no fp8 copy (xs8 is None); want_xs False: no bf16 copy (xs is
    None: fp8 experts whose weight gradients are in fp8 too never read it)."""
    return native.tfb_moe_gather(h2, tab, x_scale, want_xs)


def moe_mlp8_fwd(xs8, w8, rows, tab, F):
    """Grouped fp8 expert MLP forward: (ys bf16 [rmax,d], r bf16 [rmax,F]). w8 uint8 [E,4,F*d], rows fp32 [E,16]."""
    return native.tfb_moe_mlp8_fwd(xs8, w8, rows, tab, F)


def moe_mlp_fwd(xs, w_fc, w_proj, tab):
    """Grouped bf16 expert MLP forward: (ys bf16 [rmax,d], r bf16 [rmax,F] = relu(pre), h bf16 [rmax,F] = r^2).
    w_fc bf16 [E,F,d], w_proj bf16 [E,d,F]."""
    return native.tfb_moe_mlp_fwd(xs, w_fc, w_proj, tab)


def moe_mlp_bwd(dys, r, w_fc, w_proj, tab):
    """Grouped bf16 expert MLP backward: (dxs bf16 [rmax,d], dpre bf16 [rmax,F])."""
    return native.tfb_moe_mlp_bwd(dys, r, w_fc, w_proj, tab)


def moe_backward_scales(dys, rows, tab):
    _chk(dys), _chk(rows, torch.float32)
    E = rows.shape[0]
    out = torch.empty_like(rows)
    scratch = torch.empty(E, dtype=torch.int32, device=dys.device)
    _lib.call("tfb_moe_backward_scales", _p(dys), _p(tab["tile_expert"]), _p(rows), _p(out), _p(scratch), dys.shape[0],
              dys.shape[1], E, _stream())
    return out


def moe_backward_scales_rowmax(rowmax, rows, tab, d):
    """moe_backward_scales from the row maxima moe_combine_bwd(..., want_rowmax=True) left: the same rows, no pass over dys."""
    return native.tfb_moe_backward_scales_rowmax(rowmax, rows, tab, d)


def moe_quant(x, rows, col, fmt, tab):
    """fp8 bytes of x [rmax,d] at its rows' experts' scales rows[expert][col]; rows that no expert has are zero."""
    return native.tfb_moe_quant(x, rows, col, fmt, tab)


def moe_quant_dout(dout, gate, rows, tab):
    """moe_quant(dys, rows, 5, FMT_E5M2, tab) of the dys that moe_combine_bwd writes, from dout itself."""
    return native.tfb_moe_quant_dout(dout, gate, rows, tab)


def moe_mlp8_bwd(dys, r, w8, rows_bwd, tab):
    """(dxs bf16 [rmax,d], dpre bf16 [rmax,F]) from dys; rows_bwd from moe_backward_scales."""
    return native.tfb_moe_mlp8_bwd(dys, r, w8, rows_bwd, tab)


def moe_mlp8_bwd_q(dys, r, w8, rows_bwd, tab, hq_limit):
    """The grouped fp8 backward for the fp8 weight gradients: (dxs bf16 [rmax,d], dp8 e5m2 [rmax,F], hq8 e4m3 [rmax,F],
    dy8 e5m2 [rmax,d]); no bf16 dpre is written."""
    dy8 = moe_quant(dys, rows_bwd, 5, FMT_E5M2, tab)
    return native.tfb_moe_mlp8_bwd_q(dy8, r, w8, rows_bwd, tab, hq_limit) + (dy8,)


def moe_dw8(xs8, dp8, hq8, dy8, rows_bwd, x_scale, tab, E, dw_fc=None, dw_proj=None, accumulate=False, out_dtype=bf16):
    """(dw_fc [E,F,d], dw_proj [E,d,F]) in fp8 over each expert's row segment, from the bytes the other GEMMs multiplied."""
    return native.tfb_moe_dw8(xs8, dp8, hq8, dy8, rows_bwd, x_scale, tab, E, dw_fc, dw_proj, accumulate, out_dtype == torch.float32)


def moe_dw(dpre, xs, dys, r, tab, E, dw_fc=None, dw_proj=None, accumulate=False, out_dtype=bf16):
    """(dw_fc [E,F,d], dw_proj [E,d,F]) over each expert's row segment."""
    return native.tfb_moe_dw(dpre, xs, dys, r, tab, E, dw_fc, dw_proj, accumulate, out_dtype == torch.float32)


def moe_combine(ys, tab, gate, N):
    """out [N,d]: the sum over a token's experts of its gates times their rows."""
    if gate.shape[0] != N:
        raise ValueError("gate [N, topk]")
    return native.tfb_moe_combine(ys, tab, gate)


def moe_combine_bwd(dout, ys, tab, gate, want_rowmax=False):
    """(dys, dgate), and with want_rowmax the fp32 [rmax] maxima of |dys| per row for moe_backward_scales_rowmax."""
    if want_rowmax:
        return native.tfb_moe_combine_bwd_rowmax(dout, ys, tab, gate, True)
    return native.tfb_moe_combine_bwd(dout, ys, tab, gate)


def moe_route_bwd(dgate, p, idx, dxs, tab, h2, wr, dwr=None, accumulate=False, aux=None):
    """(dh bf16 [N,d], dwr fp32 [E,d], dlogits fp32 [N,E]). aux = (terms, lse, gaux, alpha, beta): the gradient gaux
    (1-element fp32 device tensor) of the weighted auxiliary terms alpha lb + beta z of moe_aux_fwd is folded into dlogits;
    aux = (terms, lse, gaux, alpha, beta, fs, gamma, seq_len) adds the per-sequence term gamma seq of moe_aux_seq_fwd."""
    args = (dgate, p, idx, dxs, tab, h2, wr, dwr, accumulate)
    if aux is None:
        return native.tfb_moe_route_bwd(*args)
    if len(aux) == 8:
        return native.tfb_moe_route_bwd_aux_seq(*args, *aux)
    return native.tfb_moe_route_bwd_aux(*args, *aux)


def moe_aux_fwd(p, logits, tab, topk):
    """(terms fp32 [2 + E] = (lb, z, f_e), lse fp32 [N]): the router's load-balance term E sum_e f_e P_e, its z term
    mean(logsumexp(logits)^2) and the experts' load shares (round2/source/train.py:10779 moe_aux_terms)."""
    return native.tfb_moe_aux_fwd(p, logits, tab, topk)


def moe_aux_seq_fwd(p, idx, seq_len, topk):
    """(term fp32 [1], fs fp32 [N / seq_len, E]): the per-sequence balance term of moe_aux_terms
    (round2/source/train.py:10789-10792) = mean over sequences of E sum_e fs ps, and the sequences' load shares."""
    return native.tfb_moe_aux_seq_fwd(p, idx, seq_len, topk)


# ------------------------------------------------------------------------------------------ Muon Newton-Schulz
# the kit's POLAR_EXPRESS_COEFFS as the reference's kernel module holds them (round2/source/kernels/nki_nsk.py:82-88)
NS_COEFFS = (
    (8.156554524902461, -22.48329292557795, 15.878769915207462),
    (4.042929935166739, -2.808917465908714, 0.5000178451051316),
    (3.8916678022926607, -2.772484153217685, 0.5060648178503393),
    (3.285753657755655, -2.3681294933425376, 0.46449024233003106),
    (2.3465413258596377, -1.7097828382687081, 0.42323551169305323),
)
_NS_WS = {}


_NS_D_TYPES = {torch.float32: 1, bf16: 2, torch.float16: 3}


def ns5_stacks(stacks, coeffs=NS_COEFFS):
    """Five Newton-Schulz iterations on one or two stacks [(g, d), ..] whose matrices have the same long and short side: g fp32 [K, r, c]
    (tall r >= c, or wide: handled as the transposes) from X0 = bf16(bf16(g) / d), d [K] (any float dtype; the reciprocal is taken in
    fp32 as the reference's sc_tile does). Returns [(y bf16 [K, r, c], v fp32 [K, max(r, c)] = the sums of y^2 along the short side), ..]."""
    import ctypes
    if not 1 <= len(stacks) <= 2:
        raise ValueError("one or two stacks")
    M, N = max(stacks[0][0].shape[1:]), min(stacks[0][0].shape[1:])
    dev = stacks[0][0].device
    args, out, types = [], [], {d.dtype for _, d in stacks}
    d_type = _NS_D_TYPES.get(types.pop() if len(types) == 1 else None, 0)
    for g, d in stacks:
        _chk(g, torch.float32)
        K, r, c = g.shape
        if (max(r, c), min(r, c)) != (M, N):
            raise ValueError("stacks of the same long and short side")
        d = d.reshape(-1).contiguous()
        if d.numel() != K:
            raise ValueError("one denominator per matrix")
        if not d.is_cuda:
            raise RuntimeError("tfb ops need device tensors (the HIP kernels are the only implementation)")
        if g.device != dev or d.device != dev:
            raise ValueError("stacks and denominators on one device")
        d = d if d_type else d.float()
        out.append((torch.empty(K, r, c, dtype=bf16, device=g.device), torch.empty(K, M, dtype=torch.float32, device=g.device)))
        args.append((g, d, *out[-1], K, int(r < c)))
    K = sum(a[4] for a in args)
    need = _lib.lib().tfb_ns5_workspace_bytes(K, M, N)
    # one workspace per (device, stream), grown to the largest call seen (never one per shape) and kept: two stacks hold both stacks' at once,
    # twice what each alone needs
    key = (dev, torch.cuda.current_stream(dev).cuda_stream)
    ws = _NS_WS.get(key)
    if ws is None or ws.numel() < need:
        ws = _NS_WS[key] = torch.empty(max(need, 256), dtype=torch.uint8, device=dev)
    co = (ctypes.c_float * 15)(*[float(x) for t in coeffs for x in t])
    a, b = ([*map(_p, s[:4]), *s[4:]] for s in (args + [(None,) * 4 + (0, 0)])[:2])
    _lib.call("tfb_ns5_stacks", *a, *b, d_type or 1, co, M, N, _p(ws), ws.numel(), _stream())
    return out


def ns5(g, d, coeffs=NS_COEFFS):
    """ns5_stacks of one stack: (y, v)."""
    return ns5_stacks([(g, d)], coeffs)[0]


# ------------------------------------------------------------------------------------------ dense bf16 fused MLP
def mlp_fwd(x2, w_fc, w_proj):
    """(y [M,d], r [M,F]) bf16: y = bf16(bf16(r r) @ w_proj^T), r = bf16(relu(x2 @ w_fc^T)); w_fc [F,d], w_proj [d,F]
    (K/nki_mlp_fused.py:242). r is token-major (the reference's rT is r.t())."""
    return native.tfb_mlp_fwd(x2, w_fc, w_proj)


def mlp_bwd(dy2, r, w_fc, w_proj, want_h=True):
    """(dx [M,d], h [M,F] or None, dpre [M,F]) bf16: dpre = bf16(((dy2 @ w_proj) 2) r), h = bf16(r r), dx = bf16(dpre @ w_fc)
    (K/nki_mlp_fused.py:290 with dw_mode 0)."""
    return native.tfb_mlp_bwd(dy2, r, w_fc, w_proj, want_h)


# ------------------------------------------------------------------------------------------ gradient norm
def gradnorm(g_bf16=None, g_f32=None, clip=0.0):
    """fp32 [4] on the device: (sum of squares of g_bf16, of g_f32, the norm of both together, the clipping factor
    min(clip / (norm + 1e-6), 1), 1 when clip <= 0). Either buffer may be None (R1:1480, 1634)."""
    _chk(g_bf16), _chk(g_f32, torch.float32)
    ref = g_bf16 if g_bf16 is not None else g_f32
    if ref is None:
        raise ValueError("give at least one gradient buffer")
    out = torch.empty(4, dtype=torch.float32, device=ref.device)
    scr = _scratch(ref.device, int(_lib.lib().tfb_gradnorm_scratch_floats()))
    _lib.call("tfb_gradnorm", _p(g_bf16), 0 if g_bf16 is None else g_bf16.numel(), _p(g_f32),
              0 if g_f32 is None else g_f32.numel(), float(clip), _p(scr), _p(out), _stream())
    return out


# ------------------------------------------------------------------------------------------ mixer tail
def mix_tail_fwd(x2, lam, T, eps=2.0 ** -23):
    """(s1, xn2, inv): s1 = bf16(x2 + bf16(lam shift1(x2))) with shift1 inside sequences of T rows, xn2 = RMSNorm(s1);
    lam a 1-element fp32 device tensor (R1:7097)."""
    return native.tfb_mix_tail_fwd(x2, lam, T, eps)


def mix_tail_bwd(s1, inv, x2, lam, T, gy=None, ge=None):
    """(gx bf16 [rows,C], dlam fp32 [1]) from the gradients gy of xn2 and ge of s1 (either may be None) (R1:7145)."""
    return native.tfb_mix_tail_bwd(s1, inv, x2, lam, T, gy, ge)


# ------------------------------------------------------------------------------------------ replaced functions
# A program may put a function of its own in the place of any function here (ops.<name> = f, monkeypatch.setattr, ...): the
# autograd nodes then call that one. The native layer looks for it only while there is one.
_OWN = {name: fn for name, fn in list(globals().items()) if isinstance(fn, types.FunctionType) and not name.startswith("_")}


class _Module(types.ModuleType):
    def __setattr__(self, name, value):
        super().__setattr__(name, value)
        own = _OWN.get(name)
        if own is not None:
            _lib.REPLACED.pop(name, None)
            if value is not own:
                _lib.REPLACED[name] = value
            native.told()


sys.modules[__name__].__class__ = _Module
