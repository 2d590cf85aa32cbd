// The autograd nodes of the package: torch::autograd::Function classes over ops.hpp. A node takes any leading shape and
// keeps sizes itself, so no view nodes come between it and its neighbours. Weight gradients follow the in-place convention of
// the reference (round1/source/train.py:8463-8472): a weight with a `grad_buf` attribute gets its gradient added into that
// buffer and None is handed to autograd.
#include "nodes.hpp"
#include "wrapped.hpp"

#include <torch/csrc/autograd/custom_function.h>

namespace tfb {

using torch::autograd::AutogradContext;
using torch::autograd::Function;
using Vars = torch::autograd::variable_list;
namespace op = wrapped;

namespace {

// ------------------------------------------------------------------------------------------------------ node state
template <class S>
struct Holder : torch::CustomClassHolder {
  S v;
};
template <class S>
S& keep(AutogradContext* ctx) {
  auto h = c10::make_intrusive<Holder<S>>();
  S& v = h->v;
  ctx->saved_data["s"] = c10::IValue::make_capsule(std::move(h));
  return v;
}
template <class S>
S& kept(AutogradContext* ctx) {
  return static_cast<Holder<S>&>(*ctx->saved_data["s"].toCapsule()).v;
}

Tensor val(const OptTensor& t) { return t ? *t : Tensor(); }

at::DimVector dims(const Tensor& t) { return at::DimVector(t.sizes()); }

// An operand that belongs to another's rows may come in any shape of as many elements; its gradient goes back in that shape
// (and as the very same tensor where the shapes agree: amax partials may hang on it).
Tensor in_shape(const Tensor& t, at::IntArrayRef shape, const char* what) {
  TORCH_CHECK_VALUE(t.numel() == c10::multiply_integers(shape), what, " ", t.sizes(), " has not the elements of ", shape);
  return t.sizes() == shape ? dense(t) : dense(t).view(shape);
}
Tensor back_in_shape(const Tensor& g, at::IntArrayRef shape) { return !g.defined() || g.sizes() == shape ? g : g.reshape(shape); }

// ------------------------------------------------------------------------------------------- Python-side conventions
PyObject* interned(const char* s) { return PyUnicode_InternFromString(s); }
struct Names {
  PyObject *grad_buf = interned("grad_buf"), *grad_fresh = interned("grad_fresh"), *dw_part = interned("dw_part"),
           *amax = interned("_tfb_amax_part"), *w8 = interned("w8"), *w8t = interned("w8t"), *row = interned("row"), *rows = interned("rows"),
           *x_scale = interned("x_scale"), *limit = interned("limit"), *e4m3_limit = interned("e4m3_limit"), *dw_fp8 = interned("dw_fp8"),
           *sc = interned("sc"), *use_amax = interned("USE_AMAX_HINT"), *one_pass = interned("LM_HEAD_ONE_PASS");
};
const Names& names() {
  static const Names* n = new Names;
  return *n;
}

Tensor tensor_of(PyObject* o) {   // steals; None or nullptr: undefined
  Tensor t;
  if (o && THPVariable_Check(o)) t = THPVariable_Unpack(o);
  Py_XDECREF(o);
  return t;
}
Tensor tensor_attr(PyObject* o, PyObject* name) {
  Tensor t = tensor_of(attr(o, name));
  TORCH_CHECK(t.defined(), "state is not refreshed: call its refresh() first");
  return t;
}
bool bool_attr(PyObject* o, PyObject* name) {
  PyObject* a = attr(o, name);
  const bool v = a && PyObject_IsTrue(a) == 1;
  Py_XDECREF(a);
  return v;
}
double float_attr(PyObject* o, PyObject* name) {
  PyObject* a = attr(o, name);
  const double v = a ? PyFloat_AsDouble(a) : 0.0;
  Py_XDECREF(a);
  if (PyErr_Occurred()) {
    python_error e;
    e.persist();
    throw e;
  }
  return v;
}
Scale scale_attr(PyObject* o, PyObject* name) {   // a float, or a one-element fp32 device tensor
  PyObject* a = attr(o, name);
  Scale s;
  if (a && THPVariable_Check(a)) {
    s.dev = tensor_of(a);
    chk(s.dev, F32);
    TORCH_CHECK_VALUE(s.dev.numel() == 1, "a device activation scale is one fp32 element");
    return s;
  }
  Py_XDECREF(a);
  s.imm = float_attr(o, name);
  return s;
}

// A switch of the Python module autograd (missing: off). Under the GIL.
bool switched_on(PyObject* name) {
  static PyObject* dict = PyModule_GetDict(PyImport_ImportModule("trainium_frontier_them_bones_amd.autograd"));
  PyObject* v = PyDict_GetItem(dict, name);
  return v && PyObject_IsTrue(v) == 1;
}

struct GradBuf {
  Tensor buf;
  bool accumulate = false;
};
// The weight's in-place gradient buffer (undefined: none) and whether it holds earlier micro-steps' sums; marks it written. What
// the kernels take for granted of it is checked first: a dense device tensor, of the weight's shape and bf16 or fp32 where a GEMM writes
// it (flat: fp32 and as many elements).
GradBuf accumulate_into(const Tensor& w, bool flat = false) {
  pybind11::gil_scoped_acquire gil;
  PyRef o(THPVariable_Wrap(w), PyRef::Steal{});
  PyRef buf(attr(o.o, names().grad_buf), PyRef::Steal{});
  GradBuf g;
  if (!buf.o || buf.o == Py_None) return g;
  TORCH_CHECK_TYPE(THPVariable_Check(buf.o), "grad_buf must be a tensor, got ", Py_TYPE(buf.o)->tp_name);
  g.buf = THPVariable_Unpack(buf.o);
  chk(g.buf, flat ? F32 : g.buf.scalar_type());
  const bool fits = flat ? g.buf.numel() == w.numel() : g.buf.sizes() == w.sizes();
  TORCH_CHECK_VALUE((g.buf.scalar_type() == BF16 || g.buf.scalar_type() == F32) && fits,
                    "grad_buf must be bf16 or fp32 in the weight's shape ", w.sizes(), ", not ", g.buf.scalar_type(), " ", g.buf.sizes());
  PyRef fresh(attr(o.o, names().grad_fresh), PyRef::Steal{});
  g.accumulate = fresh.o && PyObject_IsTrue(fresh.o) == 0;
  PyObject_SetAttr(o.o, names().grad_fresh, Py_False);
  return g;
}
bool has_grad_buf(const Tensor& w) {
  pybind11::gil_scoped_acquire gil;
  PyRef o(THPVariable_Wrap(w), PyRef::Steal{});
  PyRef buf(attr(o.o, names().grad_buf), PyRef::Steal{});
  return buf.o && buf.o != Py_None;
}

// The norm's gain gradient: left as partial sums where the weight names a place for them (finished with the other norms' by
// one launch), added into the weight's gradient buffer, or returned.
struct NormBack {
  Tensor dx, gw, amax;
};
NormBack norm_backward(const Tensor& gy, const Tensor& s, const Tensor& inv, const Tensor& w, const Tensor& gs, bool want_amax) {
  Tensor part;
  GradBuf g;
  if (w.defined()) {
    {
      pybind11::gil_scoped_acquire gil;
      PyObject* o = THPVariable_Wrap(w);
      part = tensor_of(attr(o, names().dw_part));
      Py_DECREF(o);
    }
    if (!part.defined()) g = accumulate_into(w, true);
  }
  NormGrad n = op::rmsnorm_bwd(dense(gy), s, inv, w, dense(gs), g.buf, g.accumulate, part, want_amax);
  NormBack b{n.dx, {}, n.amax};
  if (w.defined() && !part.defined() && !g.buf.defined()) b.gw = n.dw.to(w.scalar_type());
  return b;
}

// out = weight gradient g^T a [N, K] of M rows, into the weight's buffer (undefined returned) or as a tensor.
Tensor weight_grad(const Tensor& w, const Tensor& g, const Tensor& a, int64_t M, int64_t N, int64_t K) {
  GradBuf gb = accumulate_into(w);
  if (gb.buf.defined()) {
    op::gemm(g, a, gb.buf, N, K, M, true, false, gb.accumulate);
    return {};
  }
  Tensor dw = make({N, K}, BF16, g);
  op::gemm(g, a, dw, N, K, M, true, false, false);
  return dw;
}

// dx and the weight gradient of y = x w^T for x of M rows, w [N, K].
std::pair<Tensor, Tensor> linear_backward(const Tensor& gy, const Tensor& x, const Tensor& w, int64_t M, int64_t N, int64_t K) {
  Tensor dx = make_like(x);
  if (any_replaced || !linear_bwd_applies(M, N, K)) {
    op::gemm(gy, w, dx, M, K, N, false, false, false);
    return {dx, weight_grad(w, gy, x, M, N, K)};
  }
  chk(gy), chk(x), chk(w);
  TORCH_CHECK_VALUE(gy.numel() == M * N && x.numel() == M * K && w.numel() == N * K, "operands of ", gy.numel(), ", ", x.numel(), " and ",
                    w.numel(), " elements for ", M, " x ", N, " x ", K);
  GradBuf gb = accumulate_into(w);
  const Tensor dw = gb.buf.defined() ? gb.buf : make({N, K}, BF16, gy);
  linear_bwd(gy, x, w, dx, dw, M, N, K, gb.accumulate);
  return {dx, gb.buf.defined() ? Tensor() : dw};
}

// The amax partials on a gradient that an fp8 MLP backward starts from, when they are still valid (else it makes a pass over it).
Tensor amax_of(const Tensor& gy, const Tensor& g2) {
  pybind11::gil_scoped_acquire gil;
  return switched_on(names().use_amax) ? tensor_of(amax_hint(gy, g2)) : Tensor();
}

void attach(const Tensor& dx, const Tensor& amax) {
  pybind11::gil_scoped_acquire gil;
  PyObject* a = THPVariable_Wrap(amax);
  attach_amax(dx, a);
  Py_DECREF(a);
}

// A tensor of like's shape and type without storage of its own (one NaN element, expanded): whoever reads it gets NaN.
Tensor nan_placeholder(const Tensor& like) {
  static std::mutex mu;
  static auto* made = new std::map<std::pair<int, int>, Tensor>;
  Tensor one;
  {
    std::lock_guard<std::mutex> lock(mu);
    Tensor& t = (*made)[{like.get_device(), static_cast<int>(like.scalar_type())}];
    if (!t.defined()) t = at::full({1}, std::nan(""), like.options());
    one = t;
  }
  return one.expand(like.sizes());
}

// ------------------------------------------------------------------------------------------------------------ norms
struct RmsNorm : Function<RmsNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, const OptTensor& w_, double eps) {
    ctx->set_materialize_grads(false);
    const Tensor x = dense(x_), w = val(w_);
    NormOut o = op::rmsnorm_fwd(x, w, eps, {});
    ctx->save_for_backward({x, o.inv, w});
    return o.y;
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    if (!g[0].defined()) return {Tensor(), Tensor(), Tensor()};
    const auto s = ctx->get_saved_variables();
    NormBack b = norm_backward(g[0], s[0], s[1], s[2], {}, false);
    return {b.dx, b.gw, Tensor()};
  }
};

struct RmsNormPass : Function<RmsNormPass> {
  static Vars forward(AutogradContext* ctx, const Tensor& x_, const OptTensor& w_, double eps, std::optional<double> y8_scale,
                      bool bytes_only) {
    ctx->set_materialize_grads(false);
    TORCH_CHECK_VALUE(y8_scale || !bytes_only, "bytes_only needs y8_scale");
    const Tensor x = dense(x_), w = val(w_);
    if (!y8_scale) {
      NormOut o = op::rmsnorm_fwd(x, w, eps, {});
      ctx->save_for_backward({x, o.inv, w});
      return {x, o.y};
    }
    NormOut o = op::rmsnorm_fwd_q(x, w, eps, {}, *y8_scale, !bytes_only);
    ctx->mark_non_differentiable({o.y8});
    ctx->save_for_backward({x, o.inv, w});
    return {x, bytes_only ? nan_placeholder(x) : o.y, o.y8};
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const Tensor gs = dense(g[0]);
    if (!g[1].defined()) return {gs, Tensor(), Tensor(), Tensor(), Tensor()};
    const auto s = ctx->get_saved_variables();
    NormBack b = norm_backward(g[1], s[0], s[1], s[2], gs, true);
    attach(b.dx, b.amax);   // an fp8 MLP whose backward receives this very tensor takes its scales from the partials
    return {b.dx, b.gw, Tensor(), Tensor(), Tensor()};
  }
};

struct AddRmsNorm : Function<AddRmsNorm> {
  static Vars forward(AutogradContext* ctx, const Tensor& x, const Tensor& res, const OptTensor& w_, double eps) {
    ctx->set_materialize_grads(false);
    const Tensor w = val(w_);
    NormOut o = op::rmsnorm_fwd(dense(x), w, eps, in_shape(res, x.sizes(), "res"));
    ctx->save_for_backward({o.s, o.inv, w});
    keep<at::DimVector>(ctx) = dims(res);
    return {o.s, o.y};
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const at::DimVector& res = kept<at::DimVector>(ctx);
    if (!g[1].defined()) return {g[0], back_in_shape(g[0], res), Tensor(), Tensor()};
    const auto s = ctx->get_saved_variables();
    NormBack b = norm_backward(g[1], s[0], s[1], s[2], g[0], false);
    return {b.dx, back_in_shape(b.dx, res), b.gw, Tensor()};
  }
};

struct BlockHead : Function<BlockHead> {
  struct S {
    bool has_skip;
    at::DimVector l1, l2, l3, x0, skip;
  };
  static Vars forward(AutogradContext* ctx, const Tensor& x_, const Tensor& x0_, const Tensor& l1, const Tensor& l2, const OptTensor& skip_,
                      const OptTensor& l3, double eps) {
    ctx->set_materialize_grads(false);
    const Tensor x = dense(x_), x0 = in_shape(x0_, x.sizes(), "x0"), skip = skip_ ? in_shape(*skip_, x.sizes(), "skip") : Tensor();
    TORCH_CHECK_TYPE(!skip_ || l3, "a skip needs its gain l3");
    auto one = [](const Tensor& t) { return t.reshape(1).to(F32); };
    const Tensor g1 = one(l1), gains = at::cat({g1, one(l2), skip.defined() ? one(*l3) : g1});   // (the third is unused without a skip)
    auto [x_new, x_norm, inv] = op::block_head_fwd(x, x0, gains, skip, eps);
    ctx->save_for_backward({x, x0, skip, x_new, inv, gains});
    keep<S>(ctx) = {skip.defined(), dims(l1), dims(l2), skip.defined() ? dims(*l3) : at::DimVector(), dims(x0_),
                    skip.defined() ? dims(*skip_) : at::DimVector()};
    return {x_new, x_norm};
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    const S& st = kept<S>(ctx);
    const Tensor gn = g[1].defined() ? dense(g[1]) : at::zeros_like(s[0]);
    HeadGrad h = op::block_head_bwd(dense(g[0]), gn, s[0], s[1], s[3], s[4], s[5], s[2]);
    auto gain = [&](int i, const at::DimVector& shape) { return h.dgains.narrow(0, i, 1).view(shape); };
    return {h.dx, back_in_shape(h.dx0, st.x0), gain(0, st.l1), gain(1, st.l2), back_in_shape(h.dskip, st.skip),
            st.has_skip ? gain(2, st.l3) : Tensor(), Tensor()};
  }
};

struct MixTail : Function<MixTail> {
  struct S {
    int64_t T;
    at::DimVector shape;
    at::ScalarType dt;
  };
  static Vars forward(AutogradContext* ctx, const Tensor& x_, const Tensor& lam, int64_t T) {
    ctx->set_materialize_grads(false);
    const Tensor x = dense(x_), lam32 = lam.reshape(1).to(F32);
    auto [s1, xn2, inv] = op::mix_tail_fwd(x, lam32, T, std::ldexp(1.0, -23));
    ctx->save_for_backward({x, s1, inv, lam32});
    keep<S>(ctx) = {T, dims(lam), lam.scalar_type()};
    return {s1, xn2};
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    if (!g[0].defined() && !g[1].defined()) return {Tensor(), Tensor(), Tensor()};
    const auto s = ctx->get_saved_variables();
    const S& st = kept<S>(ctx);
    auto [gx, dlam] = op::mix_tail_bwd(s[1], s[2], s[0], s[3], st.T, dense(g[1]), dense(g[0]));
    return {gx, dlam.to(st.dt).view(st.shape), Tensor()};
  }
};

struct Relu2 : Function<Relu2> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_) {
    const Tensor x = dense(x_);
    ctx->save_for_backward({x});
    return op::relu2(x);
  }
  static Vars backward(AutogradContext* ctx, Vars g) { return {op::relu2_bwd(ctx->get_saved_variables()[0], dense(g[0]))}; }
};

// ------------------------------------------------------------------------------------------------------ projections
struct Linear : Function<Linear> {
  struct S {
    bool has_res;
    at::DimVector res;
  };
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, const Tensor& w, const OptTensor& res) {
    const Tensor x = dense(x_);
    chk(x), chk(w);
    TORCH_CHECK_VALUE(w.dim() == 2 && last_dim(x) == w.size(1), "inner dimensions differ: ", x.size(-1), " vs ", w.size(1));
    Tensor y;
    if (res) {   // bf16(res + bf16(x @ w^T)): the residual add made in the GEMM's store (nki_attn_nr8.py:1003)
      y = op::matmul_res(x, w, in_shape(*res, with_last(x, w.size(0)), "res"), true);
    } else {
      y = make(with_last(x, w.size(0)), BF16, x);
      op::gemm(x, w, y, x.numel() / w.size(1), w.size(0), w.size(1), false, true, false);
    }
    ctx->save_for_backward({x, w});
    keep<S>(ctx) = {res.has_value(), res ? dims(*res) : at::DimVector()};
    return y;
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    const Tensor &x = s[0], &w = s[1], gy = dense(g[0]);
    const int64_t N = w.size(0), K = w.size(1), M = x.numel() / K;
    chk(gy);
    auto [dx, dw] = linear_backward(gy, x, w, M, N, K);
    const S& st = kept<S>(ctx);
    return {dx, dw, st.has_res ? back_in_shape(g[0], st.res) : Tensor()};
  }
};

struct Linear8 : Function<Linear8> {
  struct S {
    PyRef state;
    Tensor sx;         // the activation's (s, 1/s, amax), or undefined with a constant scale
    double imm = 1;    // 1 / the constant scale
    bool has_res;
    at::DimVector res;
  };
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, const Tensor& w, PyObject* state, std::optional<double> x_scale,
                        const OptTensor& x8_, const OptTensor& res) {
    const Tensor x = dense(x_);
    const auto& n = names();
    const Tensor sc = tensor_attr(state, n.sc), w8 = tensor_attr(state, n.w8);
    const bool dw8 = bool_attr(state, n.dw_fp8);
    chk(sc, F32);
    TORCH_CHECK_VALUE(w.dim() == 2 && last_dim(x) == w.size(1), "inner dimensions differ: ", x.size(-1), " vs ", w.size(1));
    TORCH_CHECK_VALUE(w8.sizes() == w.sizes() && sc.numel() >= 2, "the state holds another weight's bytes: ", w8.sizes(), " for ", w.sizes());
    const Tensor r = res ? in_shape(*res, with_last(x, w.size(0)), "res") : Tensor();
    S& st = keep<S>(ctx);
    st.state = PyRef(state);
    st.has_res = res.has_value();
    if (res) st.res = dims(*res);
    Tensor x8;
    if (!x_scale) {
      st.sx = op::amax_scale(x, float_attr(state, n.limit), -24, 40);
      x8 = op::quant_fp8(x, st.sx, 0, E4M3);
    } else {
      x8 = x8_ ? in_shape(*x8_, x.sizes(), "x8") : op::quant_fp8(x, {}, *x_scale, E4M3);
      st.imm = 1.0 / *x_scale;
    }
    Tensor y = op::gemm_fp8(x8, w8, E4M3, st.sx, sc, st.imm, r, with_last(x, w.size(0)));
    ctx->save_for_backward({dw8 ? x8 : x, w});
    return y;
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    const Tensor &xa = s[0], &w = s[1], gy = dense(g[0]);
    S& st = kept<S>(ctx);
    Tensor sc, w8t;
    bool dw8;
    {
      pybind11::gil_scoped_acquire gil;
      sc = tensor_attr(st.state.o, names().sc), w8t = tensor_attr(st.state.o, names().w8t), dw8 = bool_attr(st.state.o, names().dw_fp8);
    }
    const int64_t N = w.size(0), K = w.size(1), M = xa.numel() / K;
    const Tensor sg = op::amax_scale(gy, 57344.0 / 2.0, -40, 60);
    const Tensor g8 = op::quant_fp8(gy, sg, 0, E5M2);
    Tensor dx = op::gemm_fp8(g8, w8t, E5M2, sg, sc, 1.0, {}, xa.sizes());
    Tensor dw;
    if (dw8) {
      GradBuf gb = accumulate_into(w);
      dw = op::gemm_fp8_tn(g8, xa, E5M2, E4M3, sg, st.sx, st.imm, gb.buf, gb.accumulate, BF16);
      if (gb.buf.defined()) dw = Tensor();
    } else {
      dw = weight_grad(w, gy, xa, M, N, K);
    }
    return {dx, dw, Tensor(), Tensor(), Tensor(), st.has_res ? back_in_shape(g[0], st.res) : Tensor()};
  }
};

// -------------------------------------------------------------------------------------------------------- attention
void check_grad(const Tensor& go, int64_t n) {
  TORCH_CHECK_TYPE(go.is_cuda() && go.scalar_type() == BF16, "attention takes bf16 device tensors");
  TORCH_CHECK_VALUE(go.numel() == n, "o and do are [B, T, H, D]");
}

struct Attention : Function<Attention> {
  struct S {
    double scale;
    int64_t band;
  };
  static Tensor forward(AutogradContext* ctx, const Tensor& q_, const Tensor& k_, const Tensor& v_, double scale, int64_t band) {
    const Tensor q = dense(q_), k = dense(k_), v = dense(v_);
    auto [o, lse] = op::attention(q, k, v, scale, band);
    ctx->save_for_backward({q, k, v, o, lse});
    keep<S>(ctx) = {scale, band};
    return o;
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    const S& st = kept<S>(ctx);
    const Tensor &q = s[0], &k = s[1], &v = s[2], &o = s[3], go = dense(g[0]);
    check_grad(go, o.numel());
    // gradients in the inputs' own (contiguous [B, H, T, D]) layout: autograd keeps them as they are
    Tensor dq = make_like(q), dk = make_like(k), dv = make_like(v);
    op::attention_bwd(q, k, v, o, go.view(o.sizes()), s[4], st.scale, dq, dk, dv, st.band);
    return {dq, dk, dv, Tensor(), Tensor()};
  }
};

struct QkvDims {
  int64_t B, T, C, H, D;
  double scale;
  int64_t band = 0;
  op::Third third(const Tensor& t, int i, int64_t row) const { return {t, i, row, B, H, T, D}; }
};
QkvDims qkv_dims(const Tensor& qkv, int64_t n_head, double scale, int64_t band = 0) {
  TORCH_CHECK_TYPE(qkv.is_cuda() && qkv.scalar_type() == BF16, "attention takes bf16 device tensors");
  TORCH_CHECK_VALUE(qkv.dim() == 3 && n_head > 0 && qkv.size(2) % (3 * n_head) == 0, "qkv is [B, T, 3 heads D]");
  const int64_t C = qkv.size(2) / 3;
  return {qkv.size(0), qkv.size(1), C, n_head, C / n_head, scale, band};
}

struct RopeAttention : Function<RopeAttention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& qkv_, const Tensor& cos, const Tensor& sin, int64_t n_head, double scale) {
    const Tensor qkv = dense(qkv_);
    const QkvDims m = qkv_dims(qkv, n_head, scale);
    const int64_t rows = m.B * m.T;
    const Tensor rot = make({m.B, m.T, 2 * m.C}, BF16, qkv);
    op::rope(qkv, cos, sin, rot, rows, m.T, 2 * m.H, m.D, 3 * m.C, 2 * m.C, false);
    Tensor o = make({m.B, m.T, m.C}, BF16, qkv), lse = make({m.B, m.H, m.T}, F32, qkv);
    op::attn_fwd(m.third(rot, 0, 2 * m.C), m.third(rot, 1, 2 * m.C), m.third(qkv, 2, 3 * m.C), o, lse, scale, 0);
    ctx->save_for_backward({qkv, rot, o, lse, cos, sin});
    keep<QkvDims>(ctx) = m;
    return o;
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    const QkvDims& m = kept<QkvDims>(ctx);
    const Tensor &qkv = s[0], &rot = s[1], &cos = s[4], &sin = s[5], go = dense(g[0]);
    check_grad(go, s[2].numel());
    const int64_t R = 3 * m.C;
    Tensor dqkv = make_like(qkv);
    const bool fused = m.D == 64;   // the inverse rotation of dq, dk rides the backward kernels' stores
    op::attn_bwd(m.third(rot, 0, 2 * m.C), m.third(rot, 1, 2 * m.C), m.third(qkv, 2, R), s[2], go, m.third(dqkv, 0, R),
             m.third(dqkv, 1, R), m.third(dqkv, 2, R), s[3], fused ? cos : Tensor(), fused ? sin : Tensor(), m.scale, 0);
    if (!fused) op::rope(dqkv, cos, sin, dqkv, m.B * m.T, m.T, 2 * m.H, m.D, R, R, true);
    return {dqkv, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

struct RopeNorm : Function<RopeNorm> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, const Tensor& cos, const Tensor& sin, double eps) {
    const Tensor x = dense(x_);
    chk(x);
    TORCH_CHECK_VALUE(x.dim() == 4, "x is [B, T, H, D]");
    const int64_t T = x.size(1), H = x.size(2), D = x.size(3), rows = x.size(0) * T;
    Tensor y = make_like(x), r = make_like(x), inv = make({rows, H}, F32, x);
    op::rope_norm_fwd(x, cos, sin, r, y, inv, rows, T, H, D, H * D, eps);
    ctx->save_for_backward({r, inv, cos, sin});
    return y;
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    const Tensor gy = dense(g[0]), &r = s[0];
    const int64_t T = r.size(1), H = r.size(2), D = r.size(3);
    Tensor dx = make_like(r);
    op::rope_norm_bwd(gy, r, s[1], s[2], s[3], dx, r.size(0) * T, T, H, D, H * D, H * D);
    return {dx, Tensor(), Tensor(), Tensor()};
  }
};

struct RopeNormAttention : Function<RopeNormAttention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& qkv_, const Tensor& cos, const Tensor& sin, int64_t n_head, double scale,
                        double eps, int64_t band, bool heads) {
    const Tensor qkv = dense(qkv_);
    const QkvDims m = qkv_dims(qkv, n_head, scale, band);
    const int64_t rows = m.B * m.T, R = 2 * m.C;
    Tensor qk = make({rows, R}, BF16, qkv), r = make({rows, R}, BF16, qkv), inv = make({rows, 2 * m.H}, F32, qkv);
    op::rope_norm_fwd(qkv, cos, sin, r, qk, inv, rows, m.T, 2 * m.H, m.D, 3 * m.C, eps);
    Tensor o = heads ? make({m.B, m.T, m.H, m.D}, BF16, qkv) : make({m.B, m.T, m.C}, BF16, qkv), lse = make({m.B, m.H, m.T}, F32, qkv);
    op::attn_fwd(m.third(qk, 0, R), m.third(qk, 1, R), m.third(qkv, 2, 3 * m.C), o, lse, scale, band);
    ctx->save_for_backward({qkv, qk, r, inv, o, lse, cos, sin});
    keep<QkvDims>(ctx) = m;
    return o;
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    const QkvDims& m = kept<QkvDims>(ctx);
    const Tensor &qkv = s[0], &qk = s[1], go = dense(g[0]);
    check_grad(go, s[4].numel());
    const int64_t R = 2 * m.C, F = 3 * m.C;
    Tensor dqkv = make_like(qkv);
    op::attn_bwd(m.third(qk, 0, R), m.third(qk, 1, R), m.third(qkv, 2, F), s[4], go, m.third(dqkv, 0, F), m.third(dqkv, 1, F),
             m.third(dqkv, 2, F), s[5], {}, {}, m.scale, m.band);
    op::rope_norm_bwd(dqkv, s[2], s[3], s[6], s[7], dqkv, m.B * m.T, m.T, 2 * m.H, m.D, F, F);   // in place on the q and k thirds
    return {dqkv, Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

struct QkvRopeAttention : Function<QkvRopeAttention> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, const Tensor& w, const Tensor& cos, const Tensor& sin, int64_t n_head,
                        double scale) {
    const Tensor x = dense(x_);
    chk(x), chk(w);
    TORCH_CHECK_VALUE(x.dim() == 3 && w.dim() == 2 && x.size(2) == w.size(1), "x is [B, T, in], w [3C, in]");
    const int64_t B = x.size(0), T = x.size(1), C = w.size(0) / 3;
    TORCH_CHECK_VALUE(n_head > 0 && w.size(0) % (3 * n_head) == 0, "qkv is [B, T, 3 heads D]");
    const int64_t D = C / n_head;
    TORCH_CHECK_VALUE(cos.numel() >= T * (D / 2) && sin.numel() >= T * (D / 2), "cos, sin are [T, D / 2]");
    Tensor qkv;
    if (D == 64 || !any_replaced) {
      qkv = D == 64 ? op::qkv_rope(x, w, cos, sin, T, 2 * C) : qkv_rope(x, w, cos, sin, T, 2 * C, D);
    } else {   // (where an op of the package is replaced: of other heads, the ops one by one)
      qkv = make({B, T, 3 * C}, BF16, x);
      op::gemm(x, w, qkv, B * T, 3 * C, x.size(2), false, true, false);
      op::rope(qkv, cos, sin, qkv, B * T, T, 2 * n_head, D, 3 * C, 3 * C, false);
    }
    const QkvDims m = qkv_dims(qkv, n_head, scale);
    Tensor o = make({B, T, C}, BF16, x), lse = make({B, m.H, T}, F32, x);
    const int64_t R = 3 * C;
    op::attn_fwd(m.third(qkv, 0, R), m.third(qkv, 1, R), m.third(qkv, 2, R), o, lse, scale, 0);
    ctx->save_for_backward({x, w, qkv, o, lse, cos, sin});
    keep<QkvDims>(ctx) = m;
    return o;
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    const QkvDims& m = kept<QkvDims>(ctx);
    const Tensor &x = s[0], &w = s[1], &qkv = s[2], go = dense(g[0]);
    check_grad(go, s[3].numel());
    const int64_t R = 3 * m.C, K = w.size(1), M = m.B * m.T;
    const Tensor dqkv = make_like(qkv);
    const bool fused = m.D == 64;   // the inverse rotation of dq, dk rides the backward kernels' stores
    op::attn_bwd(m.third(qkv, 0, R), m.third(qkv, 1, R), m.third(qkv, 2, R), s[3], go, m.third(dqkv, 0, R), m.third(dqkv, 1, R),
             m.third(dqkv, 2, R), s[4], fused ? s[5] : Tensor(), fused ? s[6] : Tensor(), m.scale, 0);
    if (!fused) op::rope(dqkv, s[5], s[6], dqkv, M, m.T, 2 * m.H, m.D, R, R, true);
    auto [dx, dw] = linear_backward(dqkv, x, w, M, R, K);
    return {dx, dw, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

// -------------------------------------------------------------------------------------------------------------- MLP
// What the backward passes of the fp8 MLP read of the layer's state, as it stands when they run.
struct Mlp8Attrs {
  Tensor row, w8;
  Scale x_scale;
  bool dw_fp8;
  double limit;
};
Mlp8Attrs mlp8_attrs(PyObject* st) {
  const auto& n = names();
  return {tensor_attr(st, n.row), tensor_attr(st, n.w8), scale_attr(st, n.x_scale), bool_attr(st, n.dw_fp8), float_attr(st, n.e4m3_limit)};
}

// dx and the weight gradients of an fp8 MLP call from its output's gradient; xa: the bytes x8 (fp8 weight gradients) or x.
struct MlpGrads {
  Tensor dx, dw_fc, dw_proj;
};
MlpGrads mlp8_backward(const Mlp8Attrs& st, const Tensor& gy_in, const Tensor& gy, const Tensor& xa, const Tensor& r, const Tensor& w_fc,
                       const Tensor& w_proj, bool buffers) {
  const Tensor amax = amax_of(gy_in, gy);
  // (where an op of the package is replaced, the ops one by one)
  const ScaledGrad sg = any_replaced ? ScaledGrad{op::mlp8_backward_scales(gy, st.row, amax), {}, {}} : mlp8_scaled_grad(gy, st.row, amax, !st.dw_fp8);
  const Tensor& rowb = sg.row;
  const int64_t F = w_fc.size(0), d = w_fc.size(1), M = r.size(0);
  MlpGrads o;
  if (st.dw_fp8) {
    bool in_place = false;
    auto outputs = [&]() -> DwOut {
      GradBuf bf, bp;
      if (buffers) bf = accumulate_into(w_fc), bp = accumulate_into(w_proj);
      TORCH_CHECK(bf.buf.defined() == bp.buf.defined() && bf.accumulate == bp.accumulate,
                  "the fp8 weight gradients write both MLP weights' gradient buffers in one call");
      in_place = bf.buf.defined();
      o.dw_fc = bf.buf, o.dw_proj = bp.buf;
      return {bf.buf, bp.buf, bf.accumulate};
    };
    if (!any_replaced && mlp8_bwd_dw8_applies(r, d)) {
      o.dx = mlp8_bwd_dw8(gy, r, st.w8, sg, st.limit, xa, st.x_scale, [&]() -> DwOut {
        DwOut w = outputs();
        if (!in_place) w.fc = o.dw_fc = make({F, d}, BF16, gy), w.proj = o.dw_proj = make({d, F}, BF16, gy);
        return w;
      });
    } else {
      MlpBwd b = any_replaced ? op::mlp8_bwd_q(gy, r, st.w8, rowb, st.limit, false) : mlp8_bwd_q(gy, r, st.w8, sg, st.limit, false);
      const bool accumulate = outputs().accumulate;
      op::mlp8_dw8(xa, b.dp8, b.hq8, b.dy8, rowb, st.x_scale, o.dw_fc, o.dw_proj, accumulate, BF16);
      o.dx = b.dx;
    }
    if (in_place) o.dw_fc = o.dw_proj = Tensor();
    return o;
  }
  MlpBwd b = any_replaced ? op::mlp8_bwd(gy, r, st.w8, rowb, false, true) : mlp8_bwd(gy, r, st.w8, sg, false);
  o.dx = b.dx;
  if (!buffers) {
    o.dw_fc = make({F, d}, BF16, gy);
    op::gemm(b.dpre, xa, o.dw_fc, F, d, M, true, false, false);
    o.dw_proj = op::mlp_dw_proj(b.dyp, r, {}, false, BF16);
    return o;
  }
  o.dw_fc = weight_grad(w_fc, b.dpre, xa, M, F, d);
  GradBuf gp = accumulate_into(w_proj);
  o.dw_proj = op::mlp_dw_proj(b.dyp, r, gp.buf, gp.accumulate, BF16);
  if (gp.buf.defined()) o.dw_proj = Tensor();
  return o;
}

struct Mlp8 : Function<Mlp8> {
  struct S {
    PyRef state;
    bool has_res;
    at::DimVector res;
  };
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, const Tensor& w_fc, const Tensor& w_proj, PyObject* state,
                        const OptTensor& x8_, const OptTensor& res_) {
    const Mlp8Attrs st = mlp8_attrs(state);
    const Tensor x8 = x8_ ? in_shape(*x8_, x_.sizes(), "x8") : Tensor(), res = res_ ? in_shape(*res_, x_.sizes(), "res") : Tensor();
    // with the bytes given and the weight gradients in fp8 nothing reads x itself (it may be a storage-less placeholder)
    const Tensor x = x8.defined() && st.dw_fp8 ? Tensor() : dense(x_);
    MlpFwd f = op::mlp8_fwd(x, st.w8, st.row, w_fc.size(0), st.x_scale, x8, res, !st.dw_fp8);
    ctx->save_for_backward({st.dw_fp8 ? f.x8 : f.xp.defined() ? f.xp : x, f.r, w_fc, w_proj});
    S& s = keep<S>(ctx);
    s.state = PyRef(state), s.has_res = res_.has_value();
    if (res_) s.res = dims(*res_);
    return f.y;
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    S& k = kept<S>(ctx);
    Mlp8Attrs st;
    {
      pybind11::gil_scoped_acquire gil;
      st = mlp8_attrs(k.state.o);
    }
    MlpGrads m = mlp8_backward(st, g[0], dense(g[0]), s[0], s[1], s[2], s[3], true);
    return {m.dx, m.dw_fc, m.dw_proj, Tensor(), Tensor(), k.has_res ? back_in_shape(g[0], k.res) : Tensor()};
  }
};

struct NrMlp : Function<NrMlp> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, const Tensor& w_fc, const Tensor& w_proj, PyObject* state, double eps) {
    const Mlp8Attrs st = mlp8_attrs(state);
    const Tensor x = dense(x_);
    // (with the weight gradients in fp8 too nothing reads the norm's bf16 rows: only its e4m3 bytes are written)
    NormOut n = op::rmsnorm_fwd_q(x, {}, eps, {}, st.x_scale.host(), !st.dw_fp8, tile_rows(x.numel() / last_dim(x)));
    MlpFwd f = op::mlp8_fwd(n.y, st.w8, st.row, w_fc.size(0), st.x_scale, n.y8, x);
    ctx->save_for_backward({x, st.dw_fp8 ? n.y8 : n.y, n.inv, f.r, w_fc, w_proj});
    keep<PyRef>(ctx) = PyRef(state);
    return f.y;
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    Mlp8Attrs st;
    {
      pybind11::gil_scoped_acquire gil;
      st = mlp8_attrs(kept<PyRef>(ctx).o);
    }
    const Tensor gy = dense(g[0]);
    MlpGrads m = mlp8_backward(st, g[0], gy, s[1], s[3], s[4], s[5], false);
    NormGrad n = op::rmsnorm_bwd(m.dx, s[0], s[2], {}, gy, {}, false, {}, true);
    attach(n.dx, n.amax);   // for the block before this one, whose backward receives this as its dy
    return {n.dx, m.dw_fc, m.dw_proj, Tensor(), Tensor()};
  }
};

struct MlpFused : Function<MlpFused> {
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, const Tensor& w_fc, const Tensor& w_proj) {
    const Tensor x = dense(x_);
    auto [y, r] = op::mlp_fwd(x, w_fc, w_proj);
    ctx->save_for_backward({x, r, w_fc, w_proj});
    return y;
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    const Tensor gy = dense(g[0]);
    const int64_t F = s[2].size(0), d = s[2].size(1), M = s[1].size(0);
    MlpBwd b = op::mlp_bwd(gy, s[1], s[2], s[3], true);
    Tensor dw_fc = weight_grad(s[2], b.dpre, s[0], M, F, d);   // dpre^T x
    return {b.dx, dw_fc, weight_grad(s[3], gy, b.h, M, d, F)};   // dy^T h
  }
};

// ----------------------------------------------------------------------------------------------- mixture of experts
struct Moe : Function<Moe> {
  struct S {
    PyRef state;   // null: bf16 experts
    MoeTab tab;
    std::vector<double> aux;
    int64_t seq_len = 0, topk = 0;
  };
  struct Attrs {
    Tensor rows, w8;
    Scale x_scale;
    double limit = 0;
    bool dw_fp8 = false;
  };
  static Attrs attrs(PyObject* st) {
    const auto& n = names();
    return {tensor_attr(st, n.rows), tensor_attr(st, n.w8), scale_attr(st, n.x_scale), float_attr(st, n.e4m3_limit), bool_attr(st, n.dw_fp8)};
  }
  static Tensor bf(const Tensor& w) { return dense(w.scalar_type() == BF16 ? w : w.to(BF16)); }

  static Vars forward(AutogradContext* ctx, const Tensor& h_, const Tensor& router, const Tensor& w_fc, const Tensor& w_proj,
                      PyObject* state, int64_t topk, const OptTensor& bias, const std::vector<double>& aux_weights, int64_t capacity,
                      PyObject* info) {
    ctx->set_materialize_grads(false);
    const Tensor h = dense(h_);
    const int64_t E = w_fc.size(0), F = w_fc.size(1), d = w_fc.size(2);
    const Tensor wr = dense(router.scalar_type() == F32 ? router : router.to(F32));
    TORCH_CHECK_VALUE(last_dim(h) == d && wr.size(1) == d && wr.size(0) == E, "h [.., d], router [E, d], w_fc [E, F, d]");
    S& s = keep<S>(ctx);
    s.aux = aux_weights, s.topk = topk;
    MoeRoute rt = op::moe_route(h, wr, topk, val(bias), !aux_weights.empty());
    s.tab = op::moe_tables(rt.idx, E, h.dim() >= 2 ? h.size(-2) : -1, capacity);
    Tensor xs, xs8, ys, r;
    if (state) {
      s.state = PyRef(state);
      const Attrs a = attrs(state);
      std::tie(xs, xs8) = op::moe_gather(h, s.tab, &a.x_scale, !a.dw_fp8);
      std::tie(ys, r) = op::moe_mlp8_fwd(xs8, a.w8, a.rows, s.tab, F);
      if (!a.dw_fp8) xs8 = Tensor();   // only the fp8 weight gradient reads the bytes again
    } else {
      std::tie(xs, xs8) = op::moe_gather(h, s.tab, nullptr, true);
      std::tie(ys, r) = op::moe_mlp_fwd(xs, bf(w_fc), bf(w_proj), s.tab);
    }
    Tensor out = op::moe_combine(ys, s.tab, rt.gate, h.sizes());
    if (info) {
      const Tensor share = s.tab.cnt.sum().to(F32) / double(rt.idx.numel());
      PyObject* k = THPVariable_Wrap(share);
      PyDict_SetItemString(info, "kept", k);
      Py_DECREF(k);
    }
    if (aux_weights.empty()) {
      ctx->save_for_backward({h, wr, rt.p, rt.idx, rt.gate, xs, xs8, ys, r, router, w_fc, w_proj});
      return {out};
    }
    auto [terms, lse] = op::moe_aux_fwd(rt.p, rt.logits, s.tab, topk);
    Tensor aux = terms.select(0, 0) * aux_weights[0] + terms.select(0, 1) * aux_weights[1];
    Tensor fs;
    if (aux_weights.size() > 2 && aux_weights[2] != 0.0) {
      TORCH_CHECK_VALUE(h.dim() >= 3, "MoeMlp8Fn: the per-sequence balance term needs h [b, t, d]");
      s.seq_len = h.size(-2);
      Tensor term;
      std::tie(term, fs) = op::moe_aux_seq_fwd(rt.p, rt.idx, s.seq_len, topk);
      aux = aux + term.select(0, 0) * aux_weights[2];
    }
    ctx->save_for_backward({h, wr, rt.p, rt.idx, rt.gate, xs, xs8, ys, r, router, w_fc, w_proj, terms, lse, fs});
    ctx->mark_non_differentiable({terms});
    return {out, aux, terms};
  }

  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto v = ctx->get_saved_variables();
    const Tensor &h = v[0], &wr = v[1], &p = v[2], &idx = v[3], &gate = v[4], &xs = v[5], &xs8 = v[6], &ys = v[7], &r = v[8], &router = v[9],
                 &w_fc = v[10], &w_proj = v[11];
    S& s = kept<S>(ctx);
    MoeAux aux;
    if (!s.aux.empty()) {
      aux.terms = v[12], aux.lse = v[13], aux.fs = v[14];
      aux.gaux = g[1].defined() ? dense(g[1].reshape(1).to(F32)) : at::zeros({1}, v[12].options());
      aux.alpha = s.aux[0], aux.beta = s.aux[1], aux.gamma = s.aux.size() > 2 ? s.aux[2] : 0.0, aux.seq_len = s.seq_len;
    }
    const int64_t E = w_fc.size(0);
    const Tensor gout = g[0].defined() ? dense(g[0]) : at::zeros_like(h);
    Attrs a;
    if (s.state.o) {
      pybind11::gil_scoped_acquire gil;
      a = attrs(s.state.o);
    }
    CombineGrad c = op::moe_combine_bwd(gout, ys, s.tab, gate, s.state.o != nullptr, !a.dw_fp8);
    Tensor rows_b;
    MlpBwd m;
    if (s.state.o) {   // the experts' amax(dys) rides the kernel that writes dys
      rows_b = op::moe_backward_scales_rowmax(c.rowmax, a.rows, s.tab, ys.size(1));
      m = a.dw_fp8 ? op::moe_mlp8_bwd_q(c.dys, gout, gate, r, a.w8, rows_b, s.tab, a.limit) : op::moe_mlp8_bwd(c.dys, r, a.w8, rows_b, s.tab);
    } else {
      m = op::moe_mlp_bwd(c.dys, r, bf(w_fc), bf(w_proj), s.tab);
    }
    // one grouped launch writes both gradients: both weights carry a gradient buffer (in the same state) or neither does; the
    // "fresh" flags are only touched on the branch that really writes the buffers
    const bool in_place = has_grad_buf(w_fc);
    TORCH_CHECK(in_place == has_grad_buf(w_proj), "MoeMlp8Fn: give both expert weights a grad_buf, or neither");
    GradBuf bf_, bp;
    if (in_place) {
      bf_ = accumulate_into(w_fc), bp = accumulate_into(w_proj);
      TORCH_CHECK(bf_.accumulate == bp.accumulate, "MoeMlp8Fn: the two expert weights' gradient buffers are in different states");
      TORCH_CHECK_VALUE(bf_.buf.scalar_type() == bp.buf.scalar_type(), "MoeMlp8Fn: the two expert weights' gradient buffers differ in type");
    }
    Tensor dw_fc = bf_.buf, dw_proj = bp.buf;
    if (a.dw_fp8)
      op::moe_dw8(xs8, m.dp8, m.hq8, m.dy8, rows_b, a.x_scale.host(), s.tab, dw_fc, dw_proj, E, bf_.accumulate, BF16);
    else
      op::moe_dw(m.dpre, xs, c.dys, r, s.tab, dw_fc, dw_proj, E, bf_.accumulate, BF16);
    if (in_place) dw_fc = dw_proj = Tensor();
    GradBuf br = accumulate_into(router, true);
    RouteGrad rg = op::moe_route_bwd(c.dgate, p, idx, m.dx, s.tab, h, wr, br.buf, br.accumulate, s.aux.empty() ? nullptr : &aux);
    return {rg.dh, br.buf.defined() ? Tensor() : rg.dwr.to(router.scalar_type()), dw_fc, dw_proj, Tensor(), Tensor(), Tensor(), Tensor(),
            Tensor(), Tensor()};
  }
};

// -------------------------------------------------------------------------------------------------------- loss head
// When a gradient is wanted: the plain LM-head GEMM, then ONE pass over the logits that writes the row losses and leaves the
// logits' gradient for an upstream gradient of one in their place; the backward is the two gradient GEMMs, each multiplying its
// product by the upstream scalar (a device value) before its rounding. Otherwise the GEMM with the log-sum-exp in its epilogue.
struct LmHeadLoss : Function<LmHeadLoss> {
  struct S {
    bool one_pass, consumed = false;
    double softcap;
    int64_t M, d, V;
  };
  static Tensor forward(AutogradContext* ctx, const Tensor& x_, const Tensor& W, const Tensor& targets, double softcap, bool mean,
                        bool one_pass) {
    const Tensor x = dense(x_), tg = targets_of(targets);
    chk(x), chk(W);
    const int64_t d = last_dim(x), M = x.numel() / d, V = W.size(0);
    TORCH_CHECK_VALUE(W.dim() == 2 && W.size(1) == d && tg.numel() == M, "x [.., d], W [V, d], one target a row");
    const Tensor w = op::loss_row_weights(tg, mean, V);
    keep<S>(ctx) = {one_pass, false, softcap, M, d, V};
    if (one_pass) {
      Tensor dl = make({M, V}, BF16, x);
      op::gemm(x, W, dl, M, V, d, false, true, false);
      ctx->save_for_backward({x, W, dl});
      return std::get<0>(op::loss_fwd_bwd(dl, tg, w, softcap, M, V)).sum();
    }
    auto [logits, rows, lse] = op::lmhead_fwd(x, W, tg, softcap, w);
    ctx->save_for_backward({x, W, tg, logits, lse, w});
    return rows.sum();
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    S& k = kept<S>(ctx);
    const Tensor &x = s[0], &W = s[1];
    Tensor dl, alpha;
    if (k.one_pass) {
      dl = s[2];
      alpha = g[0].to(F32).reshape(1);
    } else {
      TORCH_CHECK(!k.consumed, "LmHeadLossFn: second backward through the same node (retain_graph): the saved logits were overwritten by "
                               "their gradient in the first one");
      k.consumed = true;
      dl = op::loss_bwd(s[3], s[2], s[4], s[5] * g[0].to(F32), true, k.softcap, k.M, k.V);
    }
    Tensor dx = make_like(x);
    op::gemm(dl, W, dx, k.M, k.d, k.V, false, false, false, alpha);
    GradBuf gb = accumulate_into(W);
    Tensor dw = gb.buf.defined() ? gb.buf : make({k.V, k.d}, BF16, x);
    op::gemm(dl, x, dw, k.V, k.d, k.M, true, false, gb.accumulate, alpha);
    return {dx, gb.buf.defined() ? Tensor() : dw, Tensor(), Tensor(), Tensor(), Tensor()};
  }
};

struct FusedLoss : Function<FusedLoss> {
  struct S {
    double softcap;
  };
  static Tensor forward(AutogradContext* ctx, const Tensor& logits, const Tensor& targets, double softcap) {
    const Tensor tg = targets_of(targets);
    const int64_t V = last_dim(logits), N = logits.numel() / V;
    TORCH_CHECK_VALUE(tg.numel() == N, "one target a row");
    auto [rows, lse] = op::loss_fwd(logits, tg, {}, softcap, N, V);
    ctx->save_for_backward({logits, tg, lse});
    keep<S>(ctx) = {softcap};
    return rows;
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    const int64_t V = last_dim(s[0]);
    return {op::loss_bwd(s[0], s[1], s[2], dense(g[0].to(F32)), false, kept<S>(ctx).softcap, s[0].numel() / V, V), Tensor(), Tensor()};
  }
};

// The reduced loss (sum, or mean over the rows whose target counts) as one node: the reduction is a weight per row.
struct ReducedLoss : Function<ReducedLoss> {
  struct S {
    double softcap;
  };
  static Tensor forward(AutogradContext* ctx, const Tensor& logits_, const Tensor& targets, bool mean, double softcap) {
    const Tensor logits = dense(logits_), tg = targets_of(targets);
    const int64_t V = last_dim(logits), N = logits.numel() / V;
    TORCH_CHECK_VALUE(tg.numel() == N, "one target a row");
    const Tensor w = op::loss_row_weights(tg, mean, V);
    auto [rows, lse] = op::loss_fwd(logits, tg, w, softcap, N, V);
    ctx->save_for_backward({logits, tg, lse, w});
    keep<S>(ctx) = {softcap};
    return rows.sum();
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    const int64_t V = last_dim(s[0]);
    return {op::loss_bwd(s[0], s[1], s[2], s[3] * g[0].to(F32), false, kept<S>(ctx).softcap, s[0].numel() / V, V), Tensor(), Tensor(), Tensor()};
  }
};

struct Embedding : Function<Embedding> {
  static Tensor forward(AutogradContext* ctx, const Tensor& idx, const Tensor& w) {
    ctx->save_for_backward({idx, w});
    return op::embedding_fwd(idx, w);
  }
  static Vars backward(AutogradContext* ctx, Vars g) {
    const auto s = ctx->get_saved_variables();
    GradBuf gb = accumulate_into(s[1], true);
    Tensor dw = gb.buf.defined() ? gb.buf.view(s[1].sizes()) : make(s[1].sizes(), F32, s[1]);
    if (!gb.accumulate) op::fill_f32(dw, 0.0);
    op::embedding_bwd(s[0], dense(g[0]), dw);
    return {Tensor(), gb.buf.defined() ? Tensor() : dw.to(s[1].scalar_type())};
  }
};

}  // namespace

// ------------------------------------------------------------------------------------- replaced ops (see wrapped.hpp)
bool any_replaced = false;

namespace {
PyObject* replaced_dict() {   // name -> function, kept by ops.py
  static PyObject* d = PyObject_GetAttrString(PyImport_ImportModule("trainium_frontier_them_bones_amd._lib"), "REPLACED");
  return d;
}
[[noreturn]] void throw_python() {
  python_error e;
  e.persist();
  throw e;
}
}  // namespace

PyObject* replaced_fn(const char* name) { return PyDict_GetItemString(replaced_dict(), name); }

std::vector<Tensor> call_replaced(PyObject* fn, PyObject* args) {
  PyRef a(args, PyRef::Steal{});
  PyRef r(PyObject_CallObject(fn, args), PyRef::Steal{});
  if (!r.o) throw_python();
  std::vector<Tensor> v;
  auto add = [&](PyObject* o) { v.push_back(THPVariable_Check(o) ? THPVariable_Unpack(o) : Tensor()); };
  if (PyTuple_Check(r.o))
    for (Py_ssize_t i = 0; i < PyTuple_GET_SIZE(r.o); ++i) add(PyTuple_GET_ITEM(r.o, i));
  else
    add(r.o);
  return v;
}

PyObject* to_dict(const MoeTab& t) {
  PyObject* d = PyDict_New();
  auto put = [&](const char* key, PyObject* v) {
    PyDict_SetItemString(d, key, v);
    Py_DECREF(v);
  };
  for (const auto& [key, v] : {std::pair<const char*, const Tensor&>{"cnt", t.cnt}, {"seg", t.seg}, {"tile_expert", t.tile_expert},
                               {"slot", t.slot}, {"tok", t.tok}, {"ksel", t.ksel}})
    put(key, THPVariable_Wrap(v));
  put("rmax", PyLong_FromLongLong(t.rmax));
  if (t.capped) put("cnt_all", THPVariable_Wrap(t.cnt_all)), put("capacity", PyLong_FromLongLong(t.capacity));
  return d;
}
MoeTab from_dict(PyObject* d) {
  TORCH_CHECK_TYPE(PyDict_Check(d), "the slot tables are a dict");
  auto get = [&](const char* key) {
    PyObject* v = PyDict_GetItemString(d, key);
    return v && THPVariable_Check(v) ? THPVariable_Unpack(v) : Tensor();
  };
  MoeTab t{get("cnt"), get("seg"), get("tile_expert"), get("slot"), get("tok"), get("ksel"), get("cnt_all")};
  for (const Tensor* x : {&t.cnt, &t.seg, &t.tile_expert, &t.slot, &t.tok, &t.ksel}) {
    TORCH_CHECK_TYPE(x->defined(), "the slot tables are incomplete");
    chk(*x, I32);
  }
  t.rmax = t.tok.numel();
  if (PyObject* c = PyDict_GetItemString(d, "capacity")) t.capped = true, t.capacity = PyLong_AsLongLong(c);
  return t;
}

namespace wrapped {

PyObject* py(const Tensor& t) {
  if (!t.defined()) Py_RETURN_NONE;
  return THPVariable_Wrap(t);
}
PyObject* py(const Scale& s) { return s.dev.defined() ? py(s.dev) : py(s.imm); }
PyObject* py(at::ScalarType dt) {
  static PyObject* torch = PyImport_ImportModule("torch");
  return PyObject_GetAttrString(torch, dt == F32 ? "float32" : "bfloat16");
}
PyObject* py(const Rope& r) { return r.cos.defined() ? Py_BuildValue("(NN)", py(r.cos), py(r.sin)) : py(None{}); }
PyObject* py(const Aux& x) {
  if (!x.p) return py(None{});
  const MoeAux& a = *x.p;
  if (!a.fs.defined()) return Py_BuildValue("(NNNdd)", py(a.terms), py(a.lse), py(a.gaux), a.alpha, a.beta);
  return Py_BuildValue("(NNNddNdL)", py(a.terms), py(a.lse), py(a.gaux), a.alpha, a.beta, py(a.fs), a.gamma, static_cast<long long>(a.seq_len));
}

MoeTab moe_tables(const Tensor& idx, int64_t E, int64_t seq_len, int64_t capacity) {
  if (C10_UNLIKELY(any_replaced)) {
    pybind11::gil_scoped_acquire gil;
    if (PyObject* fn = replaced_fn("moe_tables")) {
      const bool capped = capacity >= 0;
      PyRef a(Py_BuildValue("(NLNN)", py(idx), static_cast<long long>(E), capped ? py(seq_len) : py(None{}), capped ? py(capacity) : py(None{})),
              PyRef::Steal{});
      PyRef r(PyObject_CallObject(fn, a.o), PyRef::Steal{});
      if (!r.o) throw_python();
      return from_dict(r.o);
    }
  }
  return tfb::moe_tables(idx, E, seq_len, capacity);
}

}  // namespace wrapped

void attach_amax(const Tensor& t, PyObject* amax) {
  PyObject* o = THPVariable_Wrap(t);
  PyObject* hint = Py_BuildValue("(Ol)", amax, static_cast<long>(t._version()));
  PyObject_SetAttr(o, names().amax, hint);
  Py_XDECREF(hint);
  Py_DECREF(o);
}

PyObject* amax_hint(const Tensor& g, const Tensor& g2) {
  PyObject* o = THPVariable_Wrap(g);
  PyObject* hint = attr(o, names().amax);
  Py_DECREF(o);
  PyObject* am = nullptr;
  if (hint && PyTuple_Check(hint) && PyLong_AsLong(PyTuple_GET_ITEM(hint, 1)) == static_cast<long>(g._version()) &&
      g2.data_ptr() == g.data_ptr() && g2.numel() == g.numel()) {
    am = PyTuple_GET_ITEM(hint, 0);
    Py_INCREF(am);
  }
  Py_XDECREF(hint);
  return am;
}

Tensor rmsnorm_node(const Tensor& x, const OptTensor& w, double eps) { return RmsNorm::apply(x, w, eps); }
Tensors rmsnorm_pass_node(const Tensor& x, const OptTensor& w, double eps, std::optional<double> s, bool bytes_only) {
  return RmsNormPass::apply(x, w, eps, s, bytes_only);
}
Tensors add_rmsnorm_node(const Tensor& x, const Tensor& res, const OptTensor& w, double eps) { return AddRmsNorm::apply(x, res, w, eps); }
Tensors block_head_node(const Tensor& x, const Tensor& x0, const Tensor& l1, const Tensor& l2, const OptTensor& skip, const OptTensor& l3,
                        double eps) {
  return BlockHead::apply(x, x0, l1, l2, skip, l3, eps);
}
Tensors mix_tail_node(const Tensor& x, const Tensor& lam, int64_t T) { return MixTail::apply(x, lam, T); }
Tensor relu2_node(const Tensor& x) { return Relu2::apply(x); }
Tensor linear_node(const Tensor& x, const Tensor& w, const OptTensor& res) { return Linear::apply(x, w, res); }
Tensor linear8_node(const Tensor& x, const Tensor& w, PyObject* st, std::optional<double> s, const OptTensor& x8, const OptTensor& res) {
  return Linear8::apply(x, w, st, s, x8, res);
}
Tensor attention_node(const Tensor& q, const Tensor& k, const Tensor& v, double scale, int64_t band) {
  return Attention::apply(q, k, v, scale, band);
}
Tensor rope_attention_node(const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t n_head, double scale) {
  return RopeAttention::apply(qkv, cos, sin, n_head, scale);
}
Tensor rope_norm_node(const Tensor& x, const Tensor& cos, const Tensor& sin, double eps) { return RopeNorm::apply(x, cos, sin, eps); }
Tensor rope_norm_attention_node(const Tensor& qkv, const Tensor& cos, const Tensor& sin, int64_t n_head, double scale, double eps,
                                int64_t band, bool heads) {
  return RopeNormAttention::apply(qkv, cos, sin, n_head, scale, eps, band, heads);
}
Tensor qkv_rope_attention_node(const Tensor& x, const Tensor& w, const Tensor& cos, const Tensor& sin, int64_t n_head, double scale) {
  return QkvRopeAttention::apply(x, w, cos, sin, n_head, scale);
}
Tensor mlp8_node(const Tensor& x, const Tensor& w_fc, const Tensor& w_proj, PyObject* st, const OptTensor& x8, const OptTensor& res) {
  return Mlp8::apply(x, w_fc, w_proj, st, x8, res);
}
Tensor nr_mlp_node(const Tensor& x, const Tensor& w_fc, const Tensor& w_proj, PyObject* st, double eps) {
  return NrMlp::apply(x, w_fc, w_proj, st, eps);
}
Tensor mlp_fused_node(const Tensor& x, const Tensor& w_fc, const Tensor& w_proj) { return MlpFused::apply(x, w_fc, w_proj); }
Tensors moe_node(const Tensor& h, const Tensor& router, const Tensor& w_fc, const Tensor& w_proj, PyObject* st, int64_t topk,
                 const OptTensor& bias, const std::vector<double>& aux, int64_t capacity, PyObject* info) {
  return Moe::apply(h, router, w_fc, w_proj, st, topk, bias, aux, capacity, info);
}
Tensor lm_head_loss_node(const Tensor& x, const Tensor& W, const Tensor& targets, double softcap, bool mean) {
  // the one-pass form pays when a gradient is wanted and a row of logits fits the kernel's registers
  const bool one = at::GradMode::is_enabled() && (x.requires_grad() || W.requires_grad()) && W.size(0) <= 65536 &&
                   switched_on(names().one_pass);
  return LmHeadLoss::apply(x, W, targets, softcap, mean, one);
}
Tensor fused_loss_node(const Tensor& logits, const Tensor& targets, double softcap) { return FusedLoss::apply(logits, targets, softcap); }
Tensor reduced_loss_node(const Tensor& logits, const Tensor& targets, bool mean, double softcap) {
  return ReducedLoss::apply(logits, targets, mean, softcap);
}
Tensor embedding_node(const Tensor& idx, const Tensor& w) { return Embedding::apply(idx, w); }

}  // namespace tfb
