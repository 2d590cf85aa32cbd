// Python bindings of the native host layer (module _tfb_host): the nodes under their Python class names and the tensor-level ops under
// the names of the entry points they run. Plain vectorcall functions: positional arguments, None for "not given".
#include "nodes.hpp"
#include "wrapped.hpp"

namespace tfb {

bool timed = false;

namespace {

PyObject* lib_module() {   // trainium_frontier_them_bones_amd._lib
  static PyObject* m = PyImport_ImportModule("trainium_frontier_them_bones_amd._lib");
  return m;
}
[[noreturn]] void raise_python() {
  python_error e;
  e.persist();
  throw e;
}

// ---------------------------------------------------------------------------------------------------------- arguments
struct Args {
  PyObject* const* a;
  Py_ssize_t n;

  bool has(int i) const { return i < n && a[i] != Py_None; }
  PyObject* obj(int i) const { return has(i) ? a[i] : nullptr; }
  Tensor opt(int i) const {
    if (!has(i)) return {};
    TORCH_CHECK_TYPE(THPVariable_Check(a[i]), "argument ", i + 1, " must be a tensor, got ", Py_TYPE(a[i])->tp_name);
    return THPVariable_Unpack(a[i]);
  }
  Tensor t(int i) const {
    TORCH_CHECK_TYPE(has(i), "argument ", i + 1, " (a tensor) is missing");
    return opt(i);
  }
  OptTensor maybe(int i) const { return has(i) ? OptTensor(opt(i)) : OptTensor(); }
  PyObject* need(int i) const {   // an object that is not None
    TORCH_CHECK_TYPE(has(i), "argument ", i + 1, " is missing");
    return a[i];
  }
  double f(int i) const {
    TORCH_CHECK_TYPE(has(i), "argument ", i + 1, " (a number) is missing");
    const double v = PyFloat_AsDouble(a[i]);
    if (v == -1.0 && PyErr_Occurred()) raise_python();
    return v;
  }
  double f_or(int i, double missing) const { return i < n ? f(i) : missing; }
  double cap(int i) const { return has(i) ? f(i) : 0.0; }   // a softcap: None stands for none
  int64_t i(int k) const {
    TORCH_CHECK_TYPE(has(k), "argument ", k + 1, " (a whole number) is missing");
    const int64_t v = PyLong_AsLongLong(a[k]);
    if (v == -1 && PyErr_Occurred()) raise_python();
    return v;
  }
  int64_t i_or(int k, int64_t none) const { return has(k) ? i(k) : none; }   // missing or None
  bool b(int i, bool missing = false) const {
    if (i >= n) return missing;
    const int v = PyObject_IsTrue(a[i]);
    if (v < 0) raise_python();
    return v != 0;
  }
  Scale scale(int i) const {   // a float, or a one-element fp32 device tensor
    if (!has(i) || !THPVariable_Check(a[i])) return {f(i), {}};
    const Tensor d = opt(i);
    chk(d, F32);
    TORCH_CHECK_VALUE(d.numel() == 1, "a device scale is one fp32 element");
    return {0.0, d};
  }
  at::ScalarType dtype(int i) const { return has(i) && b(i) ? F32 : BF16; }   // "fp32 output?"
  bool bthd(int i) const { return !is(i, "bhtd"); }   // a layout's name
  MoeTab tab(int i) const { return from_dict(need(i)); }
  bool is(int i, const char* s) const { return has(i) && PyUnicode_Check(a[i]) && PyUnicode_CompareWithASCIIString(a[i], s) == 0; }
};

PyObject* out(const Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
template <class... T>
PyObject* outs(const T&... t) {
  PyObject* r = PyTuple_New(sizeof...(T));
  Py_ssize_t i = 0;
  (PyTuple_SET_ITEM(r, i++, out(t)), ...);
  return r;
}
template <class... T>
PyObject* outs(const std::tuple<T...>& v) {
  return std::apply([](const auto&... t) { return outs(t...); }, v);
}
PyObject* outs(const Tensors& v) {
  PyObject* r = PyTuple_New(v.size());
  for (size_t i = 0; i < v.size(); ++i) PyTuple_SET_ITEM(r, i, out(v[i]));
  return r;
}
PyObject* none() { Py_RETURN_NONE; }

template <PyObject* (*F)(const Args&), int LO, int HI>   // a function of LO to HI arguments
PyObject* entry(PyObject*, PyObject* const* a, Py_ssize_t n) {
  HANDLE_TH_ERRORS
  TORCH_CHECK_TYPE(n >= LO && n <= HI, "takes ", LO, LO == HI ? "" : " to " + std::to_string(HI), " arguments (", n, " given)");
  return F({a, n});
  END_HANDLE_TH_ERRORS
}

// -------------------------------------------------------------------------------------------------------------- nodes
PyObject* py_rmsnorm(const Args& a) { return out(rmsnorm_node(a.t(0), a.maybe(1), a.f(2))); }
PyObject* py_rmsnorm_pass(const Args& a) {
  return outs(rmsnorm_pass_node(a.t(0), a.maybe(1), a.f(2), a.has(3) ? std::optional<double>(a.f(3)) : std::nullopt, a.b(4)));
}
PyObject* py_add_rmsnorm(const Args& a) { return outs(add_rmsnorm_node(a.t(0), a.t(1), a.maybe(2), a.f(3))); }
PyObject* py_block_head(const Args& a) {
  return outs(block_head_node(a.t(0), a.t(1), a.t(2), a.t(3), a.maybe(4), a.maybe(5), a.f(6)));
}
PyObject* py_mix_tail(const Args& a) { return outs(mix_tail_node(a.t(0), a.t(1), a.i(2))); }
PyObject* py_relu2(const Args& a) { return out(relu2_node(a.t(0))); }
PyObject* py_linear(const Args& a) { return out(linear_node(a.t(0), a.t(1), a.maybe(2))); }
PyObject* py_linear8(const Args& a) {
  return out(linear8_node(a.t(0), a.t(1), a.need(2), a.has(3) ? std::optional<double>(a.f(3)) : std::nullopt, a.maybe(4), a.maybe(5)));
}
PyObject* py_attention(const Args& a) { return out(attention_node(a.t(0), a.t(1), a.t(2), a.f(3), a.i_or(4, 0))); }
PyObject* py_rope_attention(const Args& a) { return out(rope_attention_node(a.t(0), a.t(1), a.t(2), a.i(3), a.f(4))); }
PyObject* py_rope_norm(const Args& a) { return out(rope_norm_node(a.t(0), a.t(1), a.t(2), a.f(3))); }
template <bool HEADS>
PyObject* py_rope_norm_attention(const Args& a) {
  return out(rope_norm_attention_node(a.t(0), a.t(1), a.t(2), a.i(3), a.f(4), a.f(5), a.i_or(6, 0), HEADS));
}
PyObject* py_qkv_rope_attention(const Args& a) { return out(qkv_rope_attention_node(a.t(0), a.t(1), a.t(2), a.t(3), a.i(4), a.f(5))); }
PyObject* py_mlp8(const Args& a) { return out(mlp8_node(a.t(0), a.t(1), a.t(2), a.need(3), a.maybe(4), a.maybe(5))); }
PyObject* py_nr_mlp(const Args& a) { return out(nr_mlp_node(a.t(0), a.t(1), a.t(2), a.need(3), a.f_or(4, std::ldexp(1.0, -23)))); }
PyObject* py_mlp_fused(const Args& a) { return out(mlp_fused_node(a.t(0), a.t(1), a.t(2))); }
PyObject* py_moe(const Args& a) {
  std::vector<double> aux;
  if (a.has(7)) {
    const Py_ssize_t n = PySequence_Size(a.a[7]);
    if (n < 0) raise_python();
    for (Py_ssize_t k = 0; k < n; ++k) {
      PyObject* o = PySequence_GetItem(a.a[7], k);
      aux.push_back(o ? PyFloat_AsDouble(o) : 0.0);
      Py_XDECREF(o);
      if (PyErr_Occurred()) raise_python();
    }
  }
  Tensors r = moe_node(a.t(0), a.t(1), a.t(2), a.t(3), a.obj(4), a.i(5), a.maybe(6), aux, a.i_or(8, -1), a.obj(9));
  return r.size() == 1 ? out(r[0]) : outs(r);
}
PyObject* py_lm_head_loss(const Args& a) {
  return out(lm_head_loss_node(a.t(0), a.t(1), a.t(2), a.cap(3), a.is(4, "mean")));
}
PyObject* py_fused_loss(const Args& a) { return out(fused_loss_node(a.t(0), a.t(1), a.cap(2))); }
PyObject* py_reduced_loss(const Args& a) { return out(reduced_loss_node(a.t(0), a.t(1), a.b(2), a.cap(3))); }
PyObject* py_embedding(const Args& a) { return out(embedding_node(a.t(0), a.t(1))); }
PyObject* py_attach_amax(const Args& a) {
  attach_amax(a.t(0), a.need(1));
  return none();
}
PyObject* py_amax_hint(const Args& a) {
  PyObject* r = amax_hint(a.t(0), a.t(1));
  return r ? r : none();
}

// ---------------------------------------------------------------------------------------------------------------- ops
PyObject* op_gemm(const Args& a) { return out(matmul(a.t(0), a.t(1), a.b(2), a.b(3), a.opt(4), a.b(5), a.dtype(6), a.opt(7))); }
PyObject* op_gemm_res(const Args& a) { return out(matmul_res(a.t(0), a.t(1), a.t(2), a.b(3))); }
PyObject* op_qkv_rope(const Args& a) { return out(qkv_rope(a.t(0), a.t(1), a.t(2), a.t(3), a.i(4), a.i(5))); }
PyObject* op_rmsnorm_fwd(const Args& a) {
  NormOut o = rmsnorm_fwd(a.t(0), a.opt(1), a.f(2), a.opt(3));
  return outs(o.s, o.y, o.inv);
}
PyObject* op_rmsnorm_fwd_q(const Args& a) {
  NormOut o = rmsnorm_fwd_q(a.t(0), a.opt(1), a.f(2), a.opt(3), a.f(4), a.b(5), a.n > 6 ? a.i(6) : 0);
  return outs(o.s, o.y, o.inv, o.y8);
}
PyObject* op_rmsnorm_bwd(const Args& a) {
  NormGrad o = rmsnorm_bwd(a.t(0), a.t(1), a.t(2), a.opt(3), a.opt(4), a.opt(5), a.b(6), a.opt(7), a.b(8));
  return a.b(8) ? outs(o.dx, o.dw, o.amax) : outs(o.dx, o.dw);
}
PyObject* op_block_head_fwd(const Args& a) { return outs(block_head_fwd(a.t(0), a.t(1), a.t(2), a.opt(3), a.f(4))); }
PyObject* op_block_head_bwd(const Args& a) {
  HeadGrad o = block_head_bwd(a.opt(0), a.t(1), a.t(2), a.t(3), a.t(4), a.t(5), a.t(6), a.opt(7));
  return outs(o.dx, o.dx0, o.dskip, o.dgains);
}
PyObject* op_mix_tail_fwd(const Args& a) { return outs(mix_tail_fwd(a.t(0), a.t(1), a.i(2), a.f(3))); }
PyObject* op_mix_tail_bwd(const Args& a) {
  return outs(mix_tail_bwd(a.t(0), a.t(1), a.t(2), a.t(3), a.i(4), a.opt(5), a.opt(6)));
}
PyObject* op_mlp8_backward_scales(const Args& a) { return out(mlp8_backward_scales(a.t(0), a.t(1), a.opt(2))); }
PyObject* op_amax_scale(const Args& a) { return out(amax_scale(a.t(0), a.f(1), a.i(2), a.i(3))); }
PyObject* op_quant_fp8(const Args& a) { return out(quant_fp8(a.t(0), a.scale(1), int(a.i(2)))); }
const void* dev_scalar(const Args& a, int i) {
  const Tensor t = a.opt(i);
  chk(t, F32);
  return ptr(t);
}
PyObject* op_gemm_fp8(const Args& a) {   // a8, b8, fmt_a, dq_a, dq_b, dq, res
  const Tensor a8 = a.t(0), b8 = a.t(1);
  TORCH_CHECK_VALUE(a8.dim() == 2 && b8.dim() == 2, "matrices expected");
  return out(gemm_fp8(a8, b8, int(a.i(2)), dev_scalar(a, 3), dev_scalar(a, 4), a.f(5), a.opt(6), {a8.size(0), b8.size(0)}));
}
PyObject* op_gemm_fp8_tn(const Args& a) {   // g8, a8, fmt_g, fmt_a, s_g, s_a, imm, out, accumulate, fp32
  return out(gemm_fp8_tn(a.t(0), a.t(1), int(a.i(2)), int(a.i(3)), dev_scalar(a, 4), dev_scalar(a, 5), a.f(6), a.opt(7), a.b(8), a.dtype(9)));
}
PyObject* op_mlp8_fwd(const Args& a) {   // x, w8, row, F, x_scale, x8, res
  MlpFwd o = mlp8_fwd(a.opt(0), a.t(1), a.t(2), a.i(3), a.scale(4), a.opt(5), a.opt(6));
  return outs(o.y, o.r, o.x8);
}
PyObject* op_mlp8_bwd(const Args& a) {
  MlpBwd o = mlp8_bwd(a.t(0), a.t(1), a.t(2), a.t(3), a.b(4));
  return outs(o.dx, o.h, o.dpre);
}
PyObject* op_mlp8_bwd_q(const Args& a) {
  MlpBwd o = mlp8_bwd_q(a.t(0), a.t(1), a.t(2), a.t(3), a.f(4), a.b(5));
  return outs(o.dx, o.dpre, o.dp8, o.hq8, o.dy8);
}
PyObject* op_mlp8_dw8(const Args& a) {   // x8, dp8, hq8, dy8, row, x_scale, dw_fc, dw_proj, accumulate, fp32
  Tensor f = a.opt(6), p = a.opt(7);
  mlp8_dw8(a.t(0), a.t(1), a.t(2), a.t(3), a.t(4), a.scale(5), f, p, a.b(8), a.dtype(9));
  return outs(f, p);
}
PyObject* op_mlp_dw_proj(const Args& a) { return out(mlp_dw_proj(a.t(0), a.t(1), a.opt(2), a.b(3), a.dtype(4))); }
PyObject* op_mlp_fwd(const Args& a) { return outs(mlp_fwd(a.t(0), a.t(1), a.t(2))); }
PyObject* op_mlp_bwd(const Args& a) {
  MlpBwd o = mlp_bwd(a.t(0), a.t(1), a.t(2), a.t(3), a.b(4));
  return outs(o.dx, o.h, o.dpre);
}
PyObject* op_relu2(const Args& a) { return out(relu2(a.t(0), a.opt(1), int(a.i(2)))); }
PyObject* op_embedding_fwd(const Args& a) { return out(embedding_fwd(a.t(0), a.t(1))); }
PyObject* op_fill(const Args& a) {
  fill_f32(a.t(0), a.f(1));
  return none();
}
PyObject* op_adamw(const Args& a) {   // p, g, m, v, step, lr, beta1, beta2, eps, weight_decay, p_bf16
  adamw(a.t(0), a.t(1), a.t(2), a.t(3), a.f(4), a.f(5), a.f(6), a.f(7), a.f(8), a.f(9), a.opt(10));
  return none();
}
PyObject* op_row_weights(const Args& a) { return out(loss_row_weights(targets_of(a.t(0)), a.b(1), a.i_or(2, 0))); }
PyObject* op_loss_fwd(const Args& a) {   // logits [N, V], targets, row_w, softcap
  const Tensor x = a.t(0);
  return outs(loss_fwd(x, targets_of(a.t(1)), a.opt(2), a.cap(3), x.size(0), x.size(1)));
}
PyObject* op_loss_fwd_bwd(const Args& a) {
  const Tensor x = a.t(0);
  return outs(loss_fwd_bwd(x, targets_of(a.t(1)), a.opt(2), a.cap(3), x.size(0), x.size(1)));
}
PyObject* op_loss_bwd(const Args& a) {   // logits, targets, lse, grow, softcap, in place
  const Tensor x = a.t(0), o = a.b(5) ? x : make_like(x);
  loss_bwd(x, targets_of(a.t(1)), a.t(2), a.t(3), o, a.cap(4), x.size(0), x.size(1));
  return out(o);
}
PyObject* op_lmhead_fwd(const Args& a) {
  return outs(lmhead_fwd(a.t(0), a.t(1), targets_of(a.t(2)), a.cap(3), a.opt(4)));
}

// attention and rotary embedding
PyObject* op_attn_fwd(const Args& a) {   // q, k, v, scale, layout, band
  return outs(attention(a.t(0), a.t(1), a.t(2), a.f(3), a.bthd(4), a.i_or(5, 0)));
}
PyObject* op_attn_bwd(const Args& a) {   // q, k, v, o, do, lse, scale, layout, dq, dk, dv, their layout, cos, sin, band
  attention_bwd(a.t(0), a.t(1), a.t(2), a.t(3), a.t(4), a.t(5), a.f(6), a.bthd(7), a.t(8), a.t(9), a.t(10), a.bthd(11), a.opt(12), a.opt(13),
                a.i_or(14, 0));
  return none();
}
PyObject* op_attn_bwd_static(const Args& a) {   // as far as the layout of dq, dk, dv
  attention_bwd_static(a.t(0), a.t(1), a.t(2), a.t(3), a.t(4), a.t(5), a.f(6), a.bthd(7), a.t(8), a.t(9), a.t(10), a.bthd(11));
  return none();
}
PyObject* op_rope(const Args& a) {   // x, cos, sin, T, heads, D, inverse, out
  const Tensor x = a.t(0), o = a.has(7) ? a.t(7) : x;
  const RowView rx = row_view(x), ro = row_view(o);
  rope(x, a.t(1), a.t(2), o, rx.rows, a.i(3), a.i(4), a.i(5), rx.stride, ro.stride, a.b(6));
  return none();
}
PyObject* op_rope_norm_fwd(const Args& a) {   // x, cos, sin, T, heads, D, eps, want_r
  const Tensor x = a.t(0);
  const RowView v = row_view(x);
  const int64_t H = a.i(4), D = a.i(5);
  Tensor y = make({v.rows, H * D}, BF16, x), r = a.b(7) ? make_like(y) : Tensor(), inv = make({v.rows, H}, F32, x);
  rope_norm_fwd(x, a.t(1), a.t(2), r, y, inv, v.rows, a.i(3), H, D, v.stride, a.f(6));
  return outs(y, r, inv);
}
PyObject* op_rope_norm_bwd(const Args& a) {   // g, r, inv, cos, sin, T, heads, D, out
  const Tensor g = a.t(0);
  const RowView v = row_view(g);
  const int64_t H = a.i(6), D = a.i(7);
  const Tensor o = a.has(8) ? a.t(8) : make({v.rows, H * D}, BF16, g);
  rope_norm_bwd(g, a.t(1), a.t(2), a.t(3), a.t(4), o, v.rows, a.i(5), H, D, v.stride, row_view(o).stride);
  return out(o);
}
PyObject* op_embedding_bwd(const Args& a) {   // idx, dy, dw
  embedding_bwd(a.t(0), a.t(1), a.t(2));
  return none();
}

// mixture of experts
PyObject* op_moe_route(const Args& a) {   // h, wr, topk, bias, want_logits
  MoeRoute o = moe_route(a.t(0), a.t(1), a.i(2), a.opt(3), a.b(4));
  return outs(o.p, o.idx, o.gate, o.logits);
}
PyObject* op_moe_tables(const Args& a) {   // idx, E, seq_len, capacity
  return to_dict(moe_tables(a.t(0), a.i(1), a.i_or(2, -1), a.i_or(3, -1)));
}
PyObject* op_moe_gather(const Args& a) {   // h, tab, x_scale, want_xs
  const Scale s = a.has(2) ? a.scale(2) : Scale{};
  return outs(moe_gather(a.t(0), a.tab(1), a.has(2) ? &s : nullptr, a.b(3)));
}
PyObject* op_moe_mlp8_fwd(const Args& a) { return outs(moe_mlp8_fwd(a.t(0), a.t(1), a.t(2), a.tab(3), a.i(4))); }
PyObject* op_moe_mlp_fwd(const Args& a) { return outs(moe_mlp_fwd(a.t(0), a.t(1), a.t(2), a.tab(3))); }
PyObject* op_moe_mlp_bwd(const Args& a) {   // dys, r, w_fc, w_proj, tab
  MlpBwd o = moe_mlp_bwd(a.t(0), a.t(1), a.t(2), a.t(3), a.tab(4));
  return outs(o.dx, o.dpre);
}
PyObject* op_moe_backward_scales_rowmax(const Args& a) { return out(moe_backward_scales_rowmax(a.t(0), a.t(1), a.tab(2), a.i(3))); }
PyObject* op_moe_quant(const Args& a) { return out(moe_quant(a.t(0), a.t(1), a.i(2), a.i(3), a.tab(4))); }
PyObject* op_moe_quant_dout(const Args& a) { return out(moe_quant_dout(a.t(0), a.t(1), a.t(2), a.tab(3))); }
PyObject* op_moe_mlp8_bwd(const Args& a) {   // dys, r, w8, rows, tab
  MlpBwd o = moe_mlp8_bwd(a.t(0), a.t(1), a.t(2), a.t(3), a.tab(4));
  return outs(o.dx, o.dpre);
}
PyObject* op_moe_mlp8_bwd_q(const Args& a) {   // dy8, r, w8, rows, tab, limit
  MlpBwd o = moe_mlp8_bwd_q(a.t(0), a.t(1), a.t(2), a.t(3), a.tab(4), a.f(5));
  return outs(o.dx, o.dp8, o.hq8);
}
PyObject* op_moe_dw8(const Args& a) {   // xs8, dp8, hq8, dy8, rows, x_scale, tab, E, dw_fc, dw_proj, accumulate, fp32
  Tensor f = a.opt(8), p = a.opt(9);
  moe_dw8(a.t(0), a.t(1), a.t(2), a.t(3), a.t(4), a.scale(5).host(), a.tab(6), f, p, a.i(7), a.b(10), a.dtype(11));
  return outs(f, p);
}
PyObject* op_moe_dw(const Args& a) {   // dpre, xs, dys, r, tab, E, dw_fc, dw_proj, accumulate, fp32
  Tensor f = a.opt(6), p = a.opt(7);
  moe_dw(a.t(0), a.t(1), a.t(2), a.t(3), a.tab(4), f, p, a.i(5), a.b(8), a.dtype(9));
  return outs(f, p);
}
PyObject* op_moe_combine(const Args& a) {   // ys, tab, gate
  const Tensor ys = a.t(0), gate = a.t(2);
  return out(moe_combine(ys, a.tab(1), gate, {gate.size(0), ys.size(1)}));
}
PyObject* op_moe_combine_bwd(const Args& a) {   // dout, ys, tab, gate, want_rowmax
  CombineGrad o = moe_combine_bwd(a.t(0), a.t(1), a.tab(2), a.t(3), a.b(4));
  return a.b(4) ? outs(o.dys, o.dgate, o.rowmax) : outs(o.dys, o.dgate);
}
PyObject* op_moe_aux_fwd(const Args& a) { return outs(moe_aux_fwd(a.t(0), a.t(1), a.tab(2), a.i(3))); }
PyObject* op_moe_aux_seq_fwd(const Args& a) { return outs(moe_aux_seq_fwd(a.t(0), a.t(1), a.i(2), a.i(3))); }
PyObject* op_moe_route_bwd(const Args& a) {
  // dgate, p, idx, dxs, tab, h, wr, dwr, accumulate[, terms, lse, gaux, alpha, beta[, fs, gamma, seq_len]]
  MoeAux x;
  if (a.n > 9) x.terms = a.t(9), x.lse = a.t(10), x.gaux = a.t(11), x.alpha = a.f(12), x.beta = a.f(13);
  if (a.n > 14) x.fs = a.t(14), x.gamma = a.f(15), x.seq_len = a.i(16);
  RouteGrad o = moe_route_bwd(a.t(0), a.t(1), a.t(2), a.t(3), a.tab(4), a.t(5), a.t(6), a.opt(7), a.b(8), a.n > 9 ? &x : nullptr);
  return outs(o.dh, o.dwr, o.dlogits);
}

PyObject* set_timed(const Args& a) {
  timed = a.b(0);
  return none();
}

PyObject* set_replaced(const Args& a) {
  any_replaced = a.b(0);
  return none();
}

// name, function, the least and the largest number of arguments
#define FN(name, f, lo, hi) \
  {name, reinterpret_cast<PyCFunction>(reinterpret_cast<void (*)()>(&entry<f, lo, hi>)), METH_FASTCALL, nullptr}
PyMethodDef methods[] = {
    FN("rmsnorm", py_rmsnorm, 3, 3), FN("rmsnorm_pass", py_rmsnorm_pass, 3, 5), FN("add_rmsnorm", py_add_rmsnorm, 4, 4),
    FN("block_head", py_block_head, 7, 7), FN("mix_tail", py_mix_tail, 3, 3), FN("relu2", py_relu2, 1, 1), FN("linear", py_linear, 2, 3),
    FN("linear8", py_linear8, 4, 6), FN("attention", py_attention, 4, 5), FN("rope_attention", py_rope_attention, 5, 5),
    FN("rope_norm", py_rope_norm, 4, 4), FN("rope_norm_attention", py_rope_norm_attention<false>, 6, 7),
    FN("rope_norm_attention_heads", py_rope_norm_attention<true>, 6, 7),
    FN("qkv_rope_attention", py_qkv_rope_attention, 6, 6), FN("mlp8", py_mlp8, 4, 6), FN("nr_mlp", py_nr_mlp, 4, 5),
    FN("mlp_fused", py_mlp_fused, 3, 3), FN("moe", py_moe, 7, 10), FN("lm_head_loss", py_lm_head_loss, 5, 5), FN("fused_loss", py_fused_loss, 3, 3),
    FN("reduced_loss", py_reduced_loss, 4, 4), FN("embedding", py_embedding, 2, 2), FN("attach_amax", py_attach_amax, 2, 2),
    FN("amax_hint", py_amax_hint, 2, 2), FN("set_timed", set_timed, 1, 1), FN("set_replaced", set_replaced, 1, 1), FN("tfb_gemm_bf16", op_gemm, 7, 7),
    FN("tfb_gemm_bf16_scaled", op_gemm, 8, 8), FN("tfb_gemm_bf16_res", op_gemm_res, 4, 4), FN("tfb_qkv_rope_fwd", op_qkv_rope, 6, 6),
    FN("tfb_rmsnorm_fwd", op_rmsnorm_fwd, 4, 4), FN("tfb_rmsnorm_fwd_q", op_rmsnorm_fwd_q, 6, 6), FN("tfb_rmsnorm_fwd_q_pad", op_rmsnorm_fwd_q, 7, 7), FN("tfb_rmsnorm_bwd", op_rmsnorm_bwd, 9, 9),
    FN("tfb_rmsnorm_bwd_amax", op_rmsnorm_bwd, 9, 9), FN("tfb_block_head_fwd", op_block_head_fwd, 5, 5),
    FN("tfb_block_head_bwd", op_block_head_bwd, 8, 8), FN("tfb_mix_tail_fwd", op_mix_tail_fwd, 4, 4), FN("tfb_mix_tail_bwd", op_mix_tail_bwd, 7, 7),
    FN("tfb_mlp8_backward_scales", op_mlp8_backward_scales, 2, 2), FN("tfb_mlp8_backward_scales_part", op_mlp8_backward_scales, 3, 3),
    FN("tfb_amax_scale", op_amax_scale, 4, 4), FN("tfb_quant_fp8", op_quant_fp8, 3, 3), FN("tfb_gemm_fp8", op_gemm_fp8, 6, 6),
    FN("tfb_gemm_fp8_res", op_gemm_fp8, 7, 7), FN("tfb_gemm_fp8_tn", op_gemm_fp8_tn, 10, 10), FN("tfb_mlp8_fwd", op_mlp8_fwd, 6, 6),
    FN("tfb_mlp8_fwd_res", op_mlp8_fwd, 7, 7), FN("tfb_mlp8_bwd", op_mlp8_bwd, 5, 5), FN("tfb_mlp8_bwd_q", op_mlp8_bwd_q, 6, 6),
    FN("tfb_mlp8_dw8", op_mlp8_dw8, 10, 10), FN("tfb_mlp_dw_proj", op_mlp_dw_proj, 5, 5), FN("tfb_mlp_fwd", op_mlp_fwd, 3, 3),
    FN("tfb_mlp_bwd", op_mlp_bwd, 5, 5), FN("tfb_relu2", op_relu2, 3, 3), FN("tfb_embedding_fwd", op_embedding_fwd, 2, 2),
    FN("tfb_fill_f32", op_fill, 2, 2), FN("tfb_adamw", op_adamw, 11, 11), FN("tfb_loss_row_weights", op_row_weights, 3, 3),
    FN("tfb_loss_fwd", op_loss_fwd, 4, 4), FN("tfb_loss_fwd_bwd", op_loss_fwd_bwd, 4, 4), FN("tfb_loss_bwd", op_loss_bwd, 6, 6),
    FN("tfb_lmhead_fwd", op_lmhead_fwd, 5, 5),
    FN("tfb_attn_fwd", op_attn_fwd, 5, 5), FN("tfb_attn_fwd_band", op_attn_fwd, 6, 6), FN("tfb_attn_bwd", op_attn_bwd, 12, 12),
    FN("tfb_attn_bwd_rope", op_attn_bwd, 14, 14), FN("tfb_attn_bwd_band", op_attn_bwd, 15, 15),
    FN("tfb_attn_bwd_static", op_attn_bwd_static, 12, 12),
    FN("tfb_rope", op_rope, 8, 8), FN("tfb_rope_norm_fwd", op_rope_norm_fwd, 8, 8), FN("tfb_rope_norm_bwd", op_rope_norm_bwd, 9, 9),
    FN("tfb_embedding_bwd_grouped", op_embedding_bwd, 3, 3), FN("tfb_moe_route", op_moe_route, 5, 5),
    FN("tfb_moe_tables", op_moe_tables, 2, 2), FN("tfb_moe_tables_cap", op_moe_tables, 4, 4), FN("tfb_moe_gather", op_moe_gather, 4, 4), FN("tfb_moe_mlp8_fwd", op_moe_mlp8_fwd, 5, 5),
    FN("tfb_moe_mlp_fwd", op_moe_mlp_fwd, 4, 4), FN("tfb_moe_mlp_bwd", op_moe_mlp_bwd, 5, 5),
    FN("tfb_moe_backward_scales_rowmax", op_moe_backward_scales_rowmax, 4, 4), FN("tfb_moe_quant", op_moe_quant, 5, 5),
    FN("tfb_moe_quant_dout", op_moe_quant_dout, 4, 4), FN("tfb_moe_mlp8_bwd", op_moe_mlp8_bwd, 5, 5),
    FN("tfb_moe_mlp8_bwd_q", op_moe_mlp8_bwd_q, 6, 6), FN("tfb_moe_dw8", op_moe_dw8, 12, 12), FN("tfb_moe_dw", op_moe_dw, 10, 10),
    FN("tfb_moe_combine", op_moe_combine, 3, 3), FN("tfb_moe_combine_bwd", op_moe_combine_bwd, 4, 4),
    FN("tfb_moe_combine_bwd_rowmax", op_moe_combine_bwd, 5, 5),
    FN("tfb_moe_aux_fwd", op_moe_aux_fwd, 4, 4), FN("tfb_moe_aux_seq_fwd", op_moe_aux_seq_fwd, 4, 4),
    FN("tfb_moe_route_bwd", op_moe_route_bwd, 9, 9), FN("tfb_moe_route_bwd_aux", op_moe_route_bwd, 14, 14),
    FN("tfb_moe_route_bwd_aux_seq", op_moe_route_bwd, 17, 17),
    {nullptr, nullptr, 0, nullptr}};
#undef FN

PyModuleDef module = {PyModuleDef_HEAD_INIT, "_tfb_host", nullptr, -1, methods, nullptr, nullptr, nullptr, nullptr};

}  // namespace

PyObject* attr(PyObject* o, PyObject* name) {
  PyObject* v = nullptr;
  if (_PyObject_LookupAttr(o, name, &v) < 0) raise_python();
  return v;
}

void raise_status(const char* name, int status) {
  pybind11::gil_scoped_acquire gil;
  PyObject* type = PyObject_GetAttrString(lib_module(), "TfbError");
  PyObject* err = type ? PyObject_CallFunction(type, "si", name, status) : nullptr;
  if (err) PyErr_SetObject(type, err);
  Py_XDECREF(err);
  Py_XDECREF(type);
  raise_python();
}

PyObject* timed_begin(const char* name) {
  PyObject* h = PyObject_CallMethod(lib_module(), "_timed_begin", "s", name);
  if (!h) raise_python();
  if (h != Py_None) return h;
  Py_DECREF(h);
  return nullptr;
}

void timed_end(PyObject* handle, const char* name, PyObject* args) {
  PyObject* r = PyObject_CallMethod(lib_module(), "_timed_end", "NsN", handle, name, args);
  if (!r) raise_python();
  Py_DECREF(r);
}

}  // namespace tfb

extern "C" __attribute__((visibility("default"))) PyObject* PyInit__tfb_host() { return PyModule_Create(&tfb::module); }
