// The ops as the autograd nodes call them. A program may put a function of its own in the place of any ops.<name> (to count calls,
// to log, to try another kernel); the nodes then call that function, with the arguments of the op, and the native one otherwise.
// While nothing is replaced a call costs one test of a flag. Names, arguments and results are those of ops.py.
#pragma once
#include <optional>
#include <string>
#include <vector>

#include "ops.hpp"

namespace tfb {

extern bool any_replaced;                                                     // some function of ops.py is not the package's own
std::vector<Tensor> call_replaced(PyObject* fn, PyObject* args);              // under the GIL; steals args; a result or a tuple of them
PyObject* replaced_fn(const char* name);                                      // what stands there instead, or nullptr; borrowed
PyObject* to_dict(const MoeTab& t);                                           // the slot tables as ops.py hands them around
MoeTab from_dict(PyObject* d);

namespace wrapped {

struct Aux { const MoeAux* p; };                                              // ops.moe_route_bwd's aux
struct Rope { const Tensor &cos, &sin; };                                     // ops.attn_bwd's rope
PyObject* py(const Tensor& t);
PyObject* py(const Scale& s);
PyObject* py(const Aux& a);
PyObject* py(const Rope& r);
PyObject* py(at::ScalarType dt);
inline PyObject* py(const MoeTab& t) { return to_dict(t); }
inline PyObject* py(double v) { return PyFloat_FromDouble(v); }
inline PyObject* py(int64_t v) { return PyLong_FromLongLong(v); }
inline PyObject* py(int v) { return PyLong_FromLong(v); }
inline PyObject* py(bool v) { return PyBool_FromLong(v); }
inline PyObject* py(const char* s) { return PyUnicode_FromString(s); }
struct None {};
inline PyObject* py(None) { Py_RETURN_NONE; }

// The results of ops.<name>(a...) where that function has been replaced.
template <class... A>
std::optional<std::vector<Tensor>> instead(const char* name, const A&... a) {
  if (C10_LIKELY(!any_replaced)) return std::nullopt;
  pybind11::gil_scoped_acquire gil;
  PyObject* fn = replaced_fn(name);
  if (!fn) return std::nullopt;
  PyObject* t = PyTuple_New(sizeof...(A));
  Py_ssize_t i = 0;
  (PyTuple_SET_ITEM(t, i++, py(a)), ...);
  std::vector<Tensor> r = call_replaced(fn, t);
  r.resize(8);                                                                // (what the function left out is undefined)
  return r;
}
inline Tensor rows(const Tensor& t, int64_t n) { return t.defined() ? t.reshape({-1, n}) : t; }

// ---- GEMM
inline void gemm(const Tensor& a, const Tensor& b, const Tensor& out, int64_t M, int64_t N, int64_t K, bool ta, bool tb, bool accumulate,
                 const Tensor& alpha = {}) {
  if (C10_UNLIKELY(any_replaced) &&
      instead("matmul", rows(a, ta ? M : K), rows(b, tb ? K : N), ta, tb, rows(out, N), accumulate, out.scalar_type(), alpha))
    return;
  tfb::gemm(a, b, out, M, N, K, ta, tb, accumulate, alpha);
}
inline Tensor matmul_res(const Tensor& a, const Tensor& b, const Tensor& res, bool tb) {
  if (auto r = instead("matmul_res", a, b, res, tb)) return (*r)[0].view(res.sizes());
  return tfb::matmul_res(a, b, res, tb);
}
inline Tensor qkv_rope(const Tensor& x, const Tensor& w, const Tensor& cos, const Tensor& sin, int64_t T, int64_t rot) {
  if (auto r = instead("qkv_rope", x, w, cos, sin, T, rot)) return (*r)[0].view(with_last(x, w.size(0)));
  return tfb::qkv_rope(x, w, cos, sin, T, rot);
}

// ---- norms
inline NormOut rmsnorm_fwd(const Tensor& x, const Tensor& w, double eps, const Tensor& res) {
  if (auto r = instead("rmsnorm_fwd", x, w, eps, res)) return {(*r)[0], (*r)[1], (*r)[2], {}};
  return tfb::rmsnorm_fwd(x, w, eps, res);
}
inline NormOut rmsnorm_fwd_q(const Tensor& x, const Tensor& w, double eps, const Tensor& res, double scale, bool want_y, int64_t rows_out = 0) {
  if (auto r = instead("rmsnorm_fwd_q", x, w, eps, res, scale, want_y, rows_out)) return {(*r)[0], (*r)[1], (*r)[2], (*r)[3]};
  return tfb::rmsnorm_fwd_q(x, w, eps, res, scale, want_y, rows_out);
}
inline NormGrad rmsnorm_bwd(const Tensor& gy, const Tensor& s, const Tensor& inv, const Tensor& w, const Tensor& gs, const Tensor& dw,
                            bool accumulate, const Tensor& part, bool want_amax) {
  if (auto r = instead("rmsnorm_bwd", gy, s, inv, w, gs, dw, accumulate, part, want_amax)) return {(*r)[0], (*r)[1], (*r)[2]};
  return tfb::rmsnorm_bwd(gy, s, inv, w, gs, dw, accumulate, part, want_amax);
}
inline std::tuple<Tensor, Tensor, Tensor> block_head_fwd(const Tensor& x, const Tensor& x0, const Tensor& gains, const Tensor& skip, double eps) {
  if (auto r = instead("block_head_fwd", x, x0, gains, skip, eps)) return {(*r)[0], (*r)[1], (*r)[2]};
  return tfb::block_head_fwd(x, x0, gains, skip, eps);
}
inline HeadGrad block_head_bwd(const Tensor& g_new, const Tensor& g_norm, const Tensor& x, const Tensor& x0, const Tensor& x_new,
                               const Tensor& inv, const Tensor& gains, const Tensor& skip) {
  if (auto r = instead("block_head_bwd", g_new, g_norm, x, x0, x_new, inv, gains, skip)) return {(*r)[0], (*r)[1], (*r)[2], (*r)[3]};
  return tfb::block_head_bwd(g_new, g_norm, x, x0, x_new, inv, gains, skip);
}
inline std::tuple<Tensor, Tensor, Tensor> mix_tail_fwd(const Tensor& x, const Tensor& lam, int64_t T, double eps) {
  if (auto r = instead("mix_tail_fwd", x, lam, T, eps)) return {(*r)[0], (*r)[1], (*r)[2]};
  return tfb::mix_tail_fwd(x, lam, T, eps);
}
inline std::tuple<Tensor, Tensor> mix_tail_bwd(const Tensor& s1, const Tensor& inv, const Tensor& x, const Tensor& lam, int64_t T,
                                               const Tensor& gy, const Tensor& ge) {
  if (auto r = instead("mix_tail_bwd", s1, inv, x, lam, T, gy, ge)) return {(*r)[0], (*r)[1]};
  return tfb::mix_tail_bwd(s1, inv, x, lam, T, gy, ge);
}

// ---- fp8
inline Tensor amax_scale(const Tensor& x, double limit, int64_t e_lo, int64_t e_hi) {
  if (auto r = instead("amax_scale", x, limit, e_lo, e_hi)) return (*r)[0];
  return tfb::amax_scale(x, limit, e_lo, e_hi);
}
// s: the (s, 1 / s, amax) that amax_scale left, or undefined with the constant scale imm
inline Tensor first(const Tensor& s, int64_t i = 0) { return s.defined() ? s.narrow(0, i, 1) : s; }
inline Tensor quant_fp8(const Tensor& x, const Tensor& s, double imm, int fmt) {
  if (C10_UNLIKELY(any_replaced))
    if (auto r = instead("quant_fp8", x, Scale{imm, first(s)}, fmt)) return (*r)[0];
  return tfb::quant_fp8(x, ptr(s), imm, fmt);
}
// sa, sb: as s above, of a8 (undefined: dq is its factor) and b8
inline Tensor gemm_fp8(const Tensor& a8, const Tensor& b8, int fmt, const Tensor& sa, const Tensor& sb, double dq, const Tensor& res,
                       at::IntArrayRef shape) {
  if (C10_UNLIKELY(any_replaced)) {
    const Tensor a = rows(a8, b8.size(1)), dqa = first(sa, 1), dqb = first(sb, 1);
    auto r = res.defined() ? instead("gemm_fp8_res", a, b8, rows(res, b8.size(0)), dqa, dqb, dq) : instead("gemm_fp8", a, b8, fmt, dqa, dqb, dq);
    if (r) return (*r)[0].view(shape);
  }
  auto inverse = [](const Tensor& s) { return s.defined() ? static_cast<const float*>(ptr(s)) + 1 : nullptr; };
  return tfb::gemm_fp8(a8, b8, fmt, inverse(sa), inverse(sb), dq, res, shape);
}
inline Tensor gemm_fp8_tn(const Tensor& g8, const Tensor& a8, int fmt_g, int fmt_a, const Tensor& sg, const Tensor& sa, double imm, const Tensor& out,
                          bool accumulate, at::ScalarType dt) {
  if (C10_UNLIKELY(any_replaced))
    if (auto r = instead("gemm_fp8_tn", rows(g8, g8.size(-1)), rows(a8, a8.size(-1)), fmt_g, fmt_a, first(sg), first(sa), imm, out, accumulate, dt))
      return (*r)[0];
  return tfb::gemm_fp8_tn(g8, a8, fmt_g, fmt_a, ptr(sg), ptr(sa), imm, out, accumulate, dt);
}

// ---- MLP
inline Tensor mlp8_backward_scales(const Tensor& dy, const Tensor& row, const Tensor& amax_part) {
  if (auto r = instead("mlp8_backward_scales", dy, row, amax_part)) return (*r)[0];
  return tfb::mlp8_backward_scales(dy, row, amax_part);
}
// x with whole tiles of rows, the others zeros
inline Tensor padded(const Tensor& x) {
  const Tensor x2 = rows(x, x.size(-1));
  return at::constant_pad_nd(x2, {0, 0, 0, tile_rows(x2.size(0)) - x2.size(0)});
}
inline MlpFwd mlp8_fwd(const Tensor& x, const Tensor& w8, const Tensor& row, int64_t F, const Scale& x_scale, const Tensor& x8, const Tensor& res,
                       bool want_xp = false) {
  if (auto r = instead("mlp8_fwd", x, w8, row, F, x_scale, true, x8, res))
    return {(*r)[0], (*r)[1], (*r)[2], want_xp && !x8.defined() ? padded(x) : Tensor()};
  return tfb::mlp8_fwd(x, w8, row, F, x_scale, x8, res, want_xp);
}
inline MlpBwd mlp8_bwd(const Tensor& dy, const Tensor& r_, const Tensor& w8, const Tensor& row, bool want_h, bool want_dyp) {
  if (auto r = instead("mlp8_bwd", dy, r_, w8, row, want_h)) {
    MlpBwd o{(*r)[0], (*r)[1], (*r)[2]};
    if (want_dyp) o.dyp = padded(dy);
    return o;
  }
  return tfb::mlp8_bwd(dy, r_, w8, row, want_h, want_dyp);
}
inline MlpBwd mlp8_bwd_q(const Tensor& dy, const Tensor& r_, const Tensor& w8, const Tensor& row, double limit, bool want_dpre) {
  if (auto r = instead("mlp8_bwd_q", dy, r_, w8, row, limit, want_dpre)) return {(*r)[0], {}, (*r)[1], (*r)[2], (*r)[3], (*r)[4], {}};
  return tfb::mlp8_bwd_q(dy, r_, w8, row, limit, want_dpre);
}
inline void mlp8_dw8(const Tensor& x8, const Tensor& dp8, const Tensor& hq8, const Tensor& dy8, const Tensor& row, const Scale& x_scale,
                     Tensor& dw_fc, Tensor& dw_proj, bool accumulate, at::ScalarType dt) {
  if (C10_UNLIKELY(any_replaced))
    if (auto r = instead("mlp8_dw8", rows(x8, x8.size(-1)), dp8, hq8, rows(dy8, dy8.size(-1)), row, x_scale, dw_fc, dw_proj, accumulate, dt)) {
      dw_fc = (*r)[0], dw_proj = (*r)[1];
      return;
    }
  tfb::mlp8_dw8(x8, dp8, hq8, dy8, row, x_scale, dw_fc, dw_proj, accumulate, dt);
}
inline Tensor mlp_dw_proj(const Tensor& dy, const Tensor& r_, const Tensor& out, bool accumulate, at::ScalarType dt) {
  if (auto r = instead("mlp_dw_proj", dy, r_, out, accumulate, dt)) return (*r)[0];
  return tfb::mlp_dw_proj(dy, r_, out, accumulate, dt);
}
inline std::tuple<Tensor, Tensor> mlp_fwd(const Tensor& x, const Tensor& w_fc, const Tensor& w_proj) {
  if (auto r = instead("mlp_fwd", x, w_fc, w_proj)) return {(*r)[0].view(x.sizes()), (*r)[1]};
  return tfb::mlp_fwd(x, w_fc, w_proj);
}
inline MlpBwd mlp_bwd(const Tensor& dy, const Tensor& r_, const Tensor& w_fc, const Tensor& w_proj, bool want_h) {
  if (auto r = instead("mlp_bwd", dy, r_, w_fc, w_proj, want_h)) return {(*r)[0], (*r)[1], (*r)[2]};
  return tfb::mlp_bwd(dy, r_, w_fc, w_proj, want_h);
}
inline Tensor relu2(const Tensor& x) {
  if (auto r = instead("relu2", x)) return (*r)[0];
  return tfb::relu2(x, {}, 0);
}
inline Tensor relu2_bwd(const Tensor& x, const Tensor& gy) {
  if (auto r = instead("relu2_bwd", x, gy)) return (*r)[0];
  return tfb::relu2(x, gy, 1);
}

// ---- attention: operands as thirds of a projection, [B, T, H, D] views of columns of `row`-element rows
struct Third {
  const Tensor& t;
  int i;
  int64_t row;
  const int64_t B, H, T, D;
  View view() const { return third(t, i, T, H * D, D, row); }
  Tensor tensor() const { return t.as_strided({B, T, H, D}, {T * row, row, D, 1}, t.storage_offset() + i * H * D); }
};
inline PyObject* py(const Third& t) { return py(t.tensor()); }
inline std::tuple<Tensor, Tensor> attention(const Tensor& q, const Tensor& k, const Tensor& v, double scale, int64_t band) {
  if (auto r = instead("attn_fwd", q, k, v, scale, "bhtd", band)) return {(*r)[0], (*r)[1]};
  return tfb::attention(q, k, v, scale, false, band);
}
inline void attention_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& go, const Tensor& lse, double scale,
                          const Tensor& dq, const Tensor& dk, const Tensor& dv, int64_t band) {
  if (instead("attn_bwd", q, k, v, o, go, lse, scale, "bhtd", dq, dk, dv, "bhtd", None{}, band)) return;
  tfb::attention_bwd(q, k, v, o, go, lse, scale, false, dq, dk, dv, false, {}, {}, band);
}
// o: any shape of [B, T, H, D]'s elements; what the call writes to when it is the native one
inline void attn_fwd(const Third& q, const Third& k, const Third& v, Tensor& o, Tensor& lse, double scale, int64_t band) {
  if (auto r = instead("attn_fwd", q, k, v, scale, "bthd", band)) {
    o = (*r)[0].view(o.sizes()), lse = (*r)[1];
    return;
  }
  tfb::attn_fwd(q.view(), k.view(), v.view(), o, lse, q.B, q.H, q.T, q.D, scale, band);
}
inline void attn_bwd(const Third& q, const Third& k, const Third& v, const Tensor& o, const Tensor& go, const Third& dq, const Third& dk,
                     const Third& dv, const Tensor& lse, const Tensor& cos, const Tensor& sin, double scale, int64_t band) {
  if (C10_UNLIKELY(any_replaced)) {
    const at::DimVector s{q.B, q.T, q.H, q.D};
    if (instead("attn_bwd", q, k, v, o.view(s), go.view(s), lse, scale, "bthd", dq, dk, dv, "bthd", Rope{cos, sin}, band)) return;
  }
  tfb::attn_bwd(q.view(), k.view(), v.view(), whole(o, q.T, q.H, q.D), whole(go, q.T, q.H, q.D), dq.view(), dk.view(), dv.view(), lse, cos, sin,
                q.B, q.H, q.T, q.D, scale, band);
}
inline void rope(const Tensor& x, const Tensor& cos, const Tensor& sin, const Tensor& out, int64_t n, int64_t T, int64_t H, int64_t D,
                 int64_t x_stride, int64_t out_stride, bool inverse) {
  if (C10_UNLIKELY(any_replaced))
    if (instead("rope_", rows(x, x_stride), cos, sin, T, H, D, inverse, rows(out, out_stride))) return;
  tfb::rope(x, cos, sin, out, n, T, H, D, x_stride, out_stride, inverse);
}
inline void rope_norm_fwd(const Tensor& x, const Tensor& cos, const Tensor& sin, Tensor& r_, Tensor& y, Tensor& inv, int64_t n, int64_t T, int64_t H,
                          int64_t D, int64_t x_stride, double eps) {
  if (C10_UNLIKELY(any_replaced))
    if (auto r = instead("rope_norm_fwd", rows(x, x_stride), cos, sin, T, H, D, eps, true)) {
      y = (*r)[0].view(y.sizes()), r_ = (*r)[1].view(r_.sizes()), inv = (*r)[2];
      return;
    }
  tfb::rope_norm_fwd(x, cos, sin, r_, y, inv, n, T, H, D, x_stride, eps);
}
inline void rope_norm_bwd(const Tensor& g, const Tensor& r_, const Tensor& inv, const Tensor& cos, const Tensor& sin, const Tensor& out, int64_t n,
                          int64_t T, int64_t H, int64_t D, int64_t g_stride, int64_t out_stride) {
  if (C10_UNLIKELY(any_replaced))
    if (instead("rope_norm_bwd", rows(g, g_stride), rows(r_, H * D), inv, cos, sin, T, H, D, rows(out, out_stride))) return;
  tfb::rope_norm_bwd(g, r_, inv, cos, sin, out, n, T, H, D, g_stride, out_stride);
}

// ---- embedding
inline Tensor embedding_fwd(const Tensor& idx, const Tensor& w) {
  if (auto r = instead("embedding_fwd", idx, w)) return (*r)[0];
  return tfb::embedding_fwd(idx, w);
}
inline void embedding_bwd(const Tensor& idx, const Tensor& dy, const Tensor& dw) {
  if (!instead("embedding_bwd", idx, dy, dw)) tfb::embedding_bwd(idx, dy, dw);
}
inline void fill_f32(const Tensor& t, double v) {
  if (!instead("fill_f32_", t, v)) tfb::fill_f32(t, v);
}

// ---- loss head (tg: what targets_of returned)
inline Tensor loss_row_weights(const Tensor& tg, bool mean, int64_t V) {
  if (auto r = instead("loss_row_weights", tg, mean ? "mean" : "sum", V)) return (*r)[0];
  return tfb::loss_row_weights(tg, mean, V);
}
inline std::tuple<Tensor, Tensor> loss_fwd(const Tensor& x, const Tensor& tg, const Tensor& row_w, double softcap, int64_t N, int64_t V) {
  if (C10_UNLIKELY(any_replaced))
    if (auto r = instead("loss_fwd", rows(x, V), tg, softcap, row_w)) return {(*r)[0], (*r)[1]};
  return tfb::loss_fwd(x, tg, row_w, softcap, N, V);
}
inline std::tuple<Tensor, Tensor> loss_fwd_bwd(const Tensor& x, const Tensor& tg, const Tensor& row_w, double softcap, int64_t N, int64_t V) {
  if (auto r = instead("loss_fwd_bwd", x, tg, row_w, softcap)) return {(*r)[0], (*r)[1]};
  return tfb::loss_fwd_bwd(x, tg, row_w, softcap, N, V);
}
// into out (undefined: in place); returns the gradient in x's shape
inline Tensor loss_bwd(const Tensor& x, const Tensor& tg, const Tensor& lse, const Tensor& grow, bool inplace, double softcap, int64_t N, int64_t V) {
  if (C10_UNLIKELY(any_replaced))
    if (auto r = instead("loss_bwd", rows(x, V), tg, lse, grow, softcap, inplace)) return (*r)[0].view(x.sizes());
  const Tensor out = inplace ? x : make_like(x);
  tfb::loss_bwd(x, tg, lse, grow, out, softcap, N, V);
  return out;
}
inline std::tuple<Tensor, Tensor, Tensor> lmhead_fwd(const Tensor& x, const Tensor& W, const Tensor& tg, double softcap, const Tensor& row_w) {
  if (auto r = instead("lmhead_fwd", x, W, tg, softcap, row_w)) return {(*r)[0], (*r)[1], (*r)[2]};
  return tfb::lmhead_fwd(x, W, tg, softcap, row_w);
}

// ---- mixture of experts
inline MoeRoute moe_route(const Tensor& h, const Tensor& wr, int64_t topk, const Tensor& bias, bool want_logits) {
  if (auto r = instead("moe_route", h, wr, topk, bias, want_logits)) return {(*r)[0], (*r)[1], (*r)[2], (*r)[3]};
  return tfb::moe_route(h, wr, topk, bias, want_logits);
}
MoeTab moe_tables(const Tensor& idx, int64_t E, int64_t seq_len, int64_t capacity);
inline std::tuple<Tensor, Tensor> moe_gather(const Tensor& h, const MoeTab& tab, const Scale* x_scale, bool want_xs) {
  if (auto r = x_scale ? instead("moe_gather", h, tab, *x_scale, want_xs) : instead("moe_gather", h, tab, None{}, want_xs))
    return {(*r)[0], (*r)[1]};
  return tfb::moe_gather(h, tab, x_scale, want_xs);
}
inline std::tuple<Tensor, Tensor> moe_mlp8_fwd(const Tensor& xs8, const Tensor& w8, const Tensor& rw, const MoeTab& tab, int64_t F) {
  if (auto r = instead("moe_mlp8_fwd", xs8, w8, rw, tab, F)) return {(*r)[0], (*r)[1]};
  return tfb::moe_mlp8_fwd(xs8, w8, rw, tab, F);
}
inline std::tuple<Tensor, Tensor> moe_mlp_fwd(const Tensor& xs, const Tensor& w_fc, const Tensor& w_proj, const MoeTab& tab) {
  if (auto r = instead("moe_mlp_fwd", xs, w_fc, w_proj, tab)) return {(*r)[0], (*r)[1]};
  auto [ys, rr, h] = tfb::moe_mlp_fwd(xs, w_fc, w_proj, tab);
  return {ys, rr};
}
inline Tensor moe_combine(const Tensor& ys, const MoeTab& tab, const Tensor& gate, at::IntArrayRef shape) {
  if (auto r = instead("moe_combine", ys, tab, gate, gate.size(0))) return (*r)[0].view(shape);
  return tfb::moe_combine(ys, tab, gate, shape);
}
// (dys is kept where some op is replaced: ops.moe_mlp8_bwd_q starts from it)
inline CombineGrad moe_combine_bwd(const Tensor& dout, const Tensor& ys, const MoeTab& tab, const Tensor& gate, bool want_rowmax, bool want_dys) {
  if (auto r = instead("moe_combine_bwd", dout, ys, tab, gate, want_rowmax)) return {(*r)[0], (*r)[1], (*r)[2]};
  return tfb::moe_combine_bwd(dout, ys, tab, gate, want_rowmax, want_dys || any_replaced);
}
inline Tensor moe_backward_scales_rowmax(const Tensor& rowmax, const Tensor& rw, const MoeTab& tab, int64_t d) {
  if (auto r = instead("moe_backward_scales_rowmax", rowmax, rw, tab, d)) return (*r)[0];
  return tfb::moe_backward_scales_rowmax(rowmax, rw, tab, d);
}
inline MlpBwd moe_mlp8_bwd(const Tensor& dys, const Tensor& r_, const Tensor& w8, const Tensor& rw, const MoeTab& tab) {
  if (auto r = instead("moe_mlp8_bwd", dys, r_, w8, rw, tab)) return {(*r)[0], {}, (*r)[1]};
  return tfb::moe_mlp8_bwd(dys, r_, w8, rw, tab);
}
// dys may be undefined while nothing is replaced: its bytes come from dout
inline MlpBwd moe_mlp8_bwd_q(const Tensor& dys, const Tensor& dout, const Tensor& gate, const Tensor& r_, const Tensor& w8, const Tensor& rw,
                             const MoeTab& tab, double limit) {
  if (dys.defined())
    if (auto r = instead("moe_mlp8_bwd_q", dys, r_, w8, rw, tab, limit)) return {(*r)[0], {}, {}, (*r)[1], (*r)[2], (*r)[3], {}};
  auto q = instead("moe_quant_dout", dout, gate, rw, tab);
  return tfb::moe_mlp8_bwd_q(q ? (*q)[0] : tfb::moe_quant_dout(dout, gate, rw, tab), r_, w8, rw, tab, limit);
}
inline MlpBwd moe_mlp_bwd(const Tensor& dys, const Tensor& r_, const Tensor& w_fc, const Tensor& w_proj, const MoeTab& tab) {
  if (auto r = instead("moe_mlp_bwd", dys, r_, w_fc, w_proj, tab)) return {(*r)[0], {}, (*r)[1]};
  return tfb::moe_mlp_bwd(dys, r_, w_fc, w_proj, tab);
}
inline void moe_dw8(const Tensor& xs8, const Tensor& dp8, const Tensor& hq8, const Tensor& dy8, const Tensor& rw, double x_scale, const MoeTab& tab,
                    Tensor& dw_fc, Tensor& dw_proj, int64_t E, bool accumulate, at::ScalarType dt) {
  if (auto r = instead("moe_dw8", xs8, dp8, hq8, dy8, rw, x_scale, tab, E, dw_fc, dw_proj, accumulate, dt)) {
    dw_fc = (*r)[0], dw_proj = (*r)[1];
    return;
  }
  tfb::moe_dw8(xs8, dp8, hq8, dy8, rw, x_scale, tab, dw_fc, dw_proj, E, accumulate, dt);
}
inline void moe_dw(const Tensor& dpre, const Tensor& xs, const Tensor& dys, const Tensor& r_, const MoeTab& tab, Tensor& dw_fc, Tensor& dw_proj,
                   int64_t E, bool accumulate, at::ScalarType dt) {
  if (auto r = instead("moe_dw", dpre, xs, dys, r_, tab, E, dw_fc, dw_proj, accumulate, dt)) {
    dw_fc = (*r)[0], dw_proj = (*r)[1];
    return;
  }
  tfb::moe_dw(dpre, xs, dys, r_, tab, dw_fc, dw_proj, E, accumulate, dt);
}
inline std::tuple<Tensor, Tensor> moe_aux_fwd(const Tensor& p, const Tensor& logits, const MoeTab& tab, int64_t topk) {
  if (auto r = instead("moe_aux_fwd", p, logits, tab, topk)) return {(*r)[0], (*r)[1]};
  return tfb::moe_aux_fwd(p, logits, tab, topk);
}
inline std::tuple<Tensor, Tensor> moe_aux_seq_fwd(const Tensor& p, const Tensor& idx, int64_t seq_len, int64_t topk) {
  if (auto r = instead("moe_aux_seq_fwd", p, idx, seq_len, topk)) return {(*r)[0], (*r)[1]};
  return tfb::moe_aux_seq_fwd(p, idx, seq_len, topk);
}
inline RouteGrad moe_route_bwd(const Tensor& dgate, const Tensor& p, const Tensor& idx, const Tensor& dxs, const MoeTab& tab, const Tensor& h,
                               const Tensor& wr, const Tensor& dwr, bool accumulate, const MoeAux* aux) {
  if (auto r = instead("moe_route_bwd", dgate, p, idx, dxs, tab, h, wr, dwr, accumulate, Aux{aux})) return {(*r)[0], (*r)[1], (*r)[2]};
  return tfb::moe_route_bwd(dgate, p, idx, dxs, tab, h, wr, dwr, accumulate, aux);
}

}  // namespace wrapped
}  // namespace tfb
