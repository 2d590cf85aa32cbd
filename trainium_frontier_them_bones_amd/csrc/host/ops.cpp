#include "ops.hpp"

#include <map>
#include <mutex>

namespace tfb {

namespace {

constexpr int64_t WORKSPACE_BYTES = 256 << 20;   // holds the largest split any entry point asks for

Tensor scratch(const Tensor& like, int64_t nfloats) { return make({nfloats}, F32, like); }

void want_shape(const Tensor& t, at::IntArrayRef s, const char* what) { TORCH_CHECK_VALUE(t.sizes() == s, what); }

struct Out2 {   // a given output is checked, a missing one made
  static Tensor get(Tensor out, at::IntArrayRef shape, at::ScalarType dt, bool accumulate, const Tensor& like) {
    if (!out.defined()) {
      TORCH_CHECK_VALUE(!accumulate, "accumulate needs out");
      return make(shape, dt, like);
    }
    chk(out, out.scalar_type());
    TORCH_CHECK_VALUE((out.scalar_type() == BF16 || out.scalar_type() == F32) && out.sizes() == shape, "bad out");
    return out;
  }
};

}  // namespace

Tensor workspace(const Tensor& like) {
  // One per (device, stream): launches on different streams would otherwise race on the same partial sums. Kept for the life of the process (streams are few: torch hands out a fixed pool).
  static std::mutex mu;
  static auto* pool = new std::map<std::pair<int, void*>, Tensor>;   // never destroyed: the device may be gone by then
  std::lock_guard<std::mutex> lock(mu);
  Tensor& ws = (*pool)[{like.get_device(), stream()}];
  if (!ws.defined()) ws = make({WORKSPACE_BYTES / 4}, F32, like);
  return ws;
}

// ---------------------------------------------------------------------------------------------------------------- GEMM
void gemm(const Tensor& a, const Tensor& b, const Tensor& out, int64_t M, int64_t N, int64_t K, bool ta, bool tb, bool accumulate,
          const Tensor& alpha) {
  chk(a), chk(b);
  TORCH_CHECK_VALUE(a.numel() == M * K && b.numel() == K * N && out.numel() == M * N, "operands of ", a.numel(), " and ", b.numel(),
                    " elements and an output of ", out.numel(), " for ", M, " x ", N, " x ", K);
  const Tensor ws = workspace(a);
  const int f32 = out.scalar_type() == F32;
  if (alpha.defined())
    TFB_CALL(tfb_gemm_bf16_scaled, ptr(a), ptr(b), ptr(out), M, N, K, ta, tb, f32, accumulate, ptr(ws), ws.numel() * 4, ptr(alpha), stream());
  else
    TFB_CALL(tfb_gemm_bf16, ptr(a), ptr(b), ptr(out), M, N, K, ta, tb, f32, accumulate, ptr(ws), ws.numel() * 4, stream());
}

bool linear_bwd_applies(int64_t M, int64_t N, int64_t K) { return M < INT32_MAX && tfb_linear_bwd_applies(M, N, K, WORKSPACE_BYTES) == 0; }

void linear_bwd(const Tensor& gy, const Tensor& x, const Tensor& w, const Tensor& dx, const Tensor& dw, int64_t M, int64_t N, int64_t K,
                bool accumulate) {
  TFB_CALL(tfb_linear_bwd, ptr(gy), ptr(x), ptr(w), ptr(dx), ptr(dw), M, N, K, dw.scalar_type() == F32, accumulate, WORKSPACE_BYTES, stream());
}

Tensor matmul(const Tensor& a, const Tensor& b, bool ta, bool tb, Tensor out, bool accumulate, at::ScalarType out_dtype, const Tensor& alpha) {
  chk(a), chk(b), chk(alpha, F32);
  TORCH_CHECK_VALUE(!alpha.defined() || alpha.numel() == 1, "alpha is one fp32 element");
  TORCH_CHECK_VALUE(a.dim() == 2 && b.dim() == 2, "matmul takes matrices");
  const int64_t M = a.size(ta), K = a.size(!ta), N = b.size(!tb);
  TORCH_CHECK_VALUE(K == b.size(tb), "inner dimensions differ: ", K, " vs ", b.size(tb));
  out = Out2::get(out, {M, N}, out_dtype, accumulate, a);
  gemm(a, b, out, M, N, K, ta, tb, accumulate, alpha);
  return out;
}

Tensor matmul_res(const Tensor& a, const Tensor& b, const Tensor& res, bool tb) {
  chk(a), chk(b), chk(res);
  TORCH_CHECK_VALUE(b.dim() == 2, "b is a matrix");
  const int64_t K = last_dim(a), M = a.numel() / K, N = b.size(!tb);
  TORCH_CHECK_VALUE(K == b.size(tb) && res.size(-1) == N && res.numel() == M * N, "shapes differ");
  Tensor out = make(res.sizes(), BF16, a);
  TFB_CALL(tfb_gemm_bf16_res, ptr(a), ptr(b), ptr(res), ptr(out), M, N, K, tb, stream());
  return out;
}

Tensor qkv_rope(const Tensor& x, const Tensor& w, const Tensor& cos, const Tensor& sin, int64_t T, int64_t rot_cols, int64_t D) {
  chk(x), chk(w), chk(cos), chk(sin);
  const int64_t K = last_dim(x), M = x.numel() / K, N = w.size(0);
  Tensor out = make(with_last(x, N), BF16, x);
  if (D == 64)
    TFB_CALL(tfb_qkv_rope_fwd, ptr(x), ptr(w), ptr(cos), ptr(sin), ptr(out), M, N, K, T, rot_cols, stream());
  else
    TFB_CALL(tfb_qkv_rope_heads_fwd, ptr(x), ptr(w), ptr(cos), ptr(sin), ptr(out), M, N, K, T, rot_cols, D, stream());
  return out;
}

// --------------------------------------------------------------------------------------------------------------- norms
NormOut rmsnorm_fwd(const Tensor& x, const Tensor& w, double eps, const Tensor& res) {
  chk(x), chk(res), chk(w);
  const int64_t C = last_dim(x), rows = x.numel() / C;
  NormOut o;
  o.y = make_like(x);
  o.s = res.defined() ? make_like(x) : x;
  o.inv = scratch(x, rows);
  TFB_CALL(tfb_rmsnorm_fwd, ptr(x), ptr(res), ptr(w), res.defined() ? ptr(o.s) : nullptr, ptr(o.y), ptr(o.inv), rows, C, eps, stream());
  return o;
}

NormOut rmsnorm_fwd_q(const Tensor& x, const Tensor& w, double eps, const Tensor& res, double y8_scale, bool want_y, int64_t rows_out) {
  chk(x), chk(res), chk(w);
  const int64_t C = last_dim(x), rows = x.numel() / C;
  NormOut o;
  const bool pad = rows_out > rows;
  if (want_y) o.y = pad ? make({rows_out, C}, BF16, x) : make_like(x);
  o.s = res.defined() ? make_like(x) : x;
  o.inv = scratch(x, rows);
  o.y8 = pad ? make({rows_out, C}, U8, x) : make(x.sizes(), U8, x);
  if (pad) {
    TFB_CALL(tfb_rmsnorm_fwd_q_pad, ptr(x), ptr(res), ptr(w), res.defined() ? ptr(o.s) : nullptr, ptr(o.y), ptr(o.inv), ptr(o.y8), y8_scale,
             rows, rows_out, C, eps, stream());
    return o;
  }
  TFB_CALL(tfb_rmsnorm_fwd_q, ptr(x), ptr(res), ptr(w), res.defined() ? ptr(o.s) : nullptr, ptr(o.y), ptr(o.inv), ptr(o.y8), y8_scale, rows,
           C, eps, stream());
  return o;
}

NormGrad rmsnorm_bwd(const Tensor& gy, const Tensor& s, const Tensor& inv, const Tensor& w, const Tensor& gs, const Tensor& dw,
                     bool accumulate, const Tensor& part_given, bool want_amax) {
  chk(gy), chk(s), chk(w), chk(gs), chk(inv, F32), chk(dw, F32), chk(part_given, F32);
  const int64_t C = last_dim(s), rows = s.numel() / C;
  const int64_t nb = w.defined() || want_amax ? tfb_norm_bwd_blocks(rows) : 0;
  TORCH_CHECK_VALUE(!dw.defined() || dw.numel() == C, "dw is [C]");
  TORCH_CHECK_VALUE(!w.defined() || !part_given.defined() || part_given.numel() >= nb * C, "part is [", nb, ", C]");
  NormGrad o;
  o.dx = make_like(s);
  Tensor part;
  if (w.defined() && part_given.defined()) {
    part = part_given;   // finished later, with the other norms', by norm_dw_finish
  } else if (w.defined()) {
    part = scratch(s, nb * C);
    o.dw = dw.defined() ? dw : scratch(s, C);
  }
  const bool acc = accumulate && dw.defined();
  if (want_amax) {
    o.amax = scratch(s, nb);
    TFB_CALL(tfb_rmsnorm_bwd_amax, ptr(gy), ptr(gs), ptr(s), ptr(w), ptr(inv), ptr(o.dx), ptr(part), ptr(o.dw), acc, ptr(o.amax), rows, C,
             stream());
  } else {
    TFB_CALL(tfb_rmsnorm_bwd, ptr(gy), ptr(gs), ptr(s), ptr(w), ptr(inv), ptr(o.dx), ptr(part), ptr(o.dw), acc, rows, C, stream());
  }
  return o;
}

std::tuple<Tensor, Tensor, Tensor> block_head_fwd(const Tensor& x, const Tensor& x0, const Tensor& gains, const Tensor& skip, double eps) {
  chk(x), chk(x0), chk(skip), chk(gains, F32);
  const int64_t C = last_dim(x), rows = x.numel() / C;
  Tensor x_new = make_like(x), x_norm = make_like(x), inv = scratch(x, rows);
  TFB_CALL(tfb_block_head_fwd, ptr(x), ptr(x0), ptr(skip), ptr(gains), ptr(x_new), ptr(x_norm), ptr(inv), rows, C, eps, stream());
  return {x_new, x_norm, inv};
}

HeadGrad block_head_bwd(const Tensor& g_new, const Tensor& g_norm, const Tensor& x, const Tensor& x0, const Tensor& x_new,
                        const Tensor& inv, const Tensor& gains, const Tensor& skip) {
  chk(g_new), chk(g_norm), chk(x), chk(x0), chk(skip), chk(x_new);
  const int64_t C = last_dim(x), rows = x.numel() / C;
  HeadGrad o{make_like(x), make_like(x), skip.defined() ? make_like(x) : Tensor(), scratch(x, 4)};
  const Tensor part = scratch(x, 4 * tfb_norm_bwd_blocks(rows));
  TFB_CALL(tfb_block_head_bwd, ptr(g_new), ptr(g_norm), ptr(x), ptr(x0), ptr(skip), ptr(x_new), ptr(inv), ptr(gains), ptr(o.dx), ptr(o.dx0),
           ptr(o.dskip), ptr(part), ptr(o.dgains), rows, C, stream());
  return o;
}

std::tuple<Tensor, Tensor, Tensor> mix_tail_fwd(const Tensor& x, const Tensor& lam, int64_t T, double eps) {
  chk(x), chk(lam, F32);
  const int64_t C = last_dim(x), rows = x.numel() / C;
  Tensor s1 = make_like(x), xn2 = make_like(x), inv = scratch(x, rows);
  TFB_CALL(tfb_mix_tail_fwd, ptr(x), ptr(lam), ptr(s1), ptr(xn2), ptr(inv), rows, C, T, eps, stream());
  return {s1, xn2, inv};
}

std::tuple<Tensor, Tensor> mix_tail_bwd(const Tensor& s1, const Tensor& inv, const Tensor& x, const Tensor& lam, int64_t T, const Tensor& gy,
                                        const Tensor& ge) {
  chk(s1), chk(x), chk(gy), chk(ge), chk(inv, F32), chk(lam, F32);
  TORCH_CHECK_VALUE(gy.defined() || ge.defined(), "give gy or ge");
  const int64_t C = last_dim(s1), rows = s1.numel() / C;
  Tensor gx = make_like(s1), part = scratch(s1, tfb_norm_bwd_blocks(rows)), dlam = scratch(s1, 1);
  TFB_CALL(tfb_mix_tail_bwd, ptr(s1), ptr(gy), ptr(ge), ptr(inv), ptr(x), ptr(lam), ptr(gx), ptr(part), ptr(dlam), rows, C, T, stream());
  return {gx, dlam};
}

// ------------------------------------------------------------------------------------------------------------- fp8 MLP
Tensor mlp8_backward_scales(const Tensor& dy, const Tensor& row, const Tensor& amax_part) {
  chk(dy), chk(row, F32), chk(amax_part, F32);
  const int64_t d = last_dim(dy), M = dy.numel() / d;
  Tensor out = scratch(dy, 16);
  if (amax_part.defined()) {
    TFB_CALL(tfb_mlp8_backward_scales_part, ptr(amax_part), amax_part.numel(), ptr(row), ptr(out), d, stream());
  } else {
    const Tensor scr = scratch(dy, 4096);
    TFB_CALL(tfb_mlp8_backward_scales, ptr(dy), ptr(row), ptr(out), ptr(scr), M, d, stream());
  }
  return out;
}

ScaledGrad mlp8_scaled_grad(const Tensor& dy, const Tensor& row, const Tensor& amax_part, bool want_padded) {
  chk(dy), chk(row, F32), chk(amax_part, F32);
  TORCH_CHECK_VALUE(row.numel() >= 16, "the scale row has ", row.numel(), " entries");
  const int64_t d = last_dim(dy), n = dy.numel(), M = tile_rows(n / d);
  ScaledGrad o{scratch(dy, 16), make({M, d}, U8, dy), want_padded && n == M * d ? dy : want_padded ? make({M, d}, BF16, dy) : Tensor()};
  const Tensor scr = amax_part.defined() ? Tensor() : scratch(dy, 4096);
  const bool copy = want_padded && n != M * d;
  TFB_CALL(tfb_mlp8_backward_quant, ptr(dy), ptr(amax_part), amax_part.defined() ? amax_part.numel() : 0, ptr(scr), ptr(row), ptr(o.row),
           ptr(o.bytes), copy ? ptr(o.padded) : nullptr, n, M * d, d, stream());
  return o;
}

Tensor amax_scale(const Tensor& x, double limit, int64_t e_lo, int64_t e_hi) {
  chk(x);
  Tensor out = scratch(x, 3), scr = scratch(x, 4096);
  TFB_CALL(tfb_amax_scale, ptr(x), x.numel(), limit, e_lo, e_hi, ptr(out), ptr(scr), stream());
  return out;
}

Tensor quant_fp8(const Tensor& x, const void* scale_dev, double scale_imm, int fmt) {
  chk(x);
  Tensor out = make(x.sizes(), U8, x);
  TFB_CALL(tfb_quant_fp8, ptr(x), scale_dev, scale_imm, fmt, ptr(out), x.numel(), stream());
  return out;
}
// The rows of x and then zeros up to M rows, as bytes; padded: the same in bf16 where x has fewer rows and it is asked for.
static Tensor quant_rows(const Tensor& x, const void* scale_dev, double scale_imm, int fmt, int64_t M, Tensor* padded) {
  const int64_t d = last_dim(x);
  if (x.numel() == M * d) {
    if (padded) *padded = x;
    return quant_fp8(x, scale_dev, scale_imm, fmt);
  }
  Tensor out = make({M, d}, U8, x);
  if (padded) *padded = make({M, d}, BF16, x);
  TFB_CALL(tfb_quant_fp8_pad, ptr(x), scale_dev, scale_imm, fmt, ptr(out), padded ? ptr(*padded) : nullptr, x.numel(), M * d, stream());
  return out;
}

// A tensor of like's shape whose storage holds M rows: the GEMM that writes it stores whole tiles.
static Tensor make_rows(at::IntArrayRef shape, int64_t M, int64_t d, const Tensor& like) {
  Tensor t = make({M, d}, BF16, like);
  t.unsafeGetTensorImpl()->set_sizes_contiguous(shape);
  return t;
}

Tensor quant_fp8(const Tensor& x, const Scale& s, int fmt) { return quant_fp8(x, ptr(s.dev), s.imm, fmt); }

Tensor gemm_fp8(const Tensor& a8, const Tensor& b8, int fmt_a, const void* dq_a, const void* dq_b, double dq, const Tensor& res,
                at::IntArrayRef out_shape) {
  chk(a8, U8), chk(b8, U8), chk(res);
  const int64_t K = last_dim(a8), M = a8.numel() / K, N = b8.size(0);
  TORCH_CHECK_VALUE(b8.dim() == 2 && b8.size(1) == K, "inner dimensions differ");
  TORCH_CHECK_VALUE(!res.defined() || (res.size(-1) == N && res.numel() == M * N), "shapes differ");
  TORCH_CHECK_VALUE(c10::multiply_integers(out_shape) == M * N, "an output ", out_shape, " for ", M, " x ", N);
  Tensor out = make(out_shape, BF16, a8);
  if (res.defined())
    TFB_CALL(tfb_gemm_fp8_res, ptr(a8), ptr(b8), dq_a, dq_b, dq, ptr(res), ptr(out), M, N, K, stream());
  else
    TFB_CALL(tfb_gemm_fp8, ptr(a8), fmt_a, ptr(b8), dq_a, dq_b, dq, ptr(out), M, N, K, stream());
  return out;
}

Tensor gemm_fp8_tn(const Tensor& g8, const Tensor& a8, int fmt_g, int fmt_a, const void* s_g, const void* s_a, double imm, Tensor out,
                   bool accumulate, at::ScalarType out_dtype) {
  chk(g8, U8), chk(a8, U8);
  const int64_t O = last_dim(g8), M = g8.numel() / O, D = last_dim(a8);
  TORCH_CHECK_VALUE(a8.numel() / D == M, "token counts differ");
  out = Out2::get(out, {O, D}, out_dtype, accumulate, g8);
  const Tensor ws = workspace(g8);
  TFB_CALL(tfb_gemm_fp8_tn, ptr(g8), fmt_g, ptr(a8), fmt_a, s_g, s_a, imm, ptr(out), M, O, D, out.scalar_type() == F32, accumulate, ptr(ws),
           ws.numel() * 4, stream());
  return out;
}

// The bytes and scale row of an MLP state are those of weights [F, d] and [d, F].
static void check_pack(const Tensor& w8, const Tensor& row, int64_t d, int64_t F) {
  TORCH_CHECK_VALUE(w8.numel() == 4 * F * d && row.numel() >= 16, "the state holds another MLP's weights: ", w8.numel(), " bytes for d ", d,
                    ", F ", F);
}

// r is what the forward of as many rows left: whole tiles where the forward padded.
static void check_rows(const Tensor& r, int64_t M, int64_t F) {
  TORCH_CHECK_VALUE(r.dim() == 2 && r.size(0) == M && r.size(1) == F, "r is [", M, ", F], not ", r.sizes());
}

MlpFwd mlp8_fwd(const Tensor& x, const Tensor& w8, const Tensor& row, int64_t F, const Scale& x_scale, const Tensor& x8, const Tensor& res,
                bool want_xp) {
  chk(x), chk(w8, U8), chk(row, F32), chk(x8, U8), chk(res);
  TORCH_CHECK_VALUE(x.defined() || x8.defined(), "give x2 or its bytes x8");
  const Tensor& in = res.defined() ? res : x.defined() ? x : x8;   // (x and x8 may come padded already, res has the call's rows)
  const int64_t d = last_dim(in), rows = in.numel() / d, M = tile_rows(rows);
  const auto fits = [&](const Tensor& t) { return t.size(-1) == d && (t.numel() == rows * d || t.numel() == M * d); };
  TORCH_CHECK_VALUE(!x8.defined() || (x8.size(-1) == d && x8.numel() == M * d), "x8 shape");
  TORCH_CHECK_VALUE(!x.defined() || fits(x), "res shape");
  check_pack(w8, row, d, F);
  MlpFwd o;
  o.x8 = x8.defined() ? x8 : quant_rows(x, ptr(x_scale.dev), x_scale.imm, E4M3, M, want_xp ? &o.xp : nullptr);
  o.y = make_rows(in.sizes(), M, d, w8);
  o.r = make({M, F}, BF16, w8);
  const Tensor h8 = make({M, F}, U8, w8);
  if (res.defined() && rows < M)
    TFB_CALL(tfb_mlp8_fwd_res_rows, ptr(o.x8), ptr(w8), ptr(row), ptr(res), ptr(o.y), ptr(o.r), ptr(h8), M, rows, d, F, stream());
  else if (res.defined())
    TFB_CALL(tfb_mlp8_fwd_res, ptr(o.x8), ptr(w8), ptr(row), ptr(res), ptr(o.y), ptr(o.r), ptr(h8), M, d, F, stream());
  else
    TFB_CALL(tfb_mlp8_fwd, ptr(o.x8), ptr(w8), ptr(row), ptr(o.y), ptr(o.r), ptr(h8), M, d, F, stream());
  return o;
}

// What a backward of dy's rows is given; the rows in whole tiles.
static int64_t check_bwd(const Tensor& dy, const Tensor& r, const Tensor& w8, const Tensor& row) {
  chk(dy), chk(r), chk(w8, U8), chk(row, F32);
  const int64_t d = last_dim(dy), M = tile_rows(dy.numel() / d), F = r.size(1);
  check_rows(r, M, F);
  check_pack(w8, row, d, F);
  return M;
}
// dy's bytes at a row's scale
static ScaledGrad at_scale(const Tensor& dy, const Tensor& row, int64_t M, bool want_padded) {
  ScaledGrad o{row, {}, {}};
  o.bytes = quant_rows(dy, static_cast<const float*>(ptr(row)) + 5, 0, E5M2, M, want_padded ? &o.padded : nullptr);
  return o;
}

MlpBwd mlp8_bwd(const Tensor& dy, const Tensor& r, const Tensor& w8, const Tensor& row, bool want_h, bool want_dyp) {
  return mlp8_bwd(dy, r, w8, at_scale(dy, row, check_bwd(dy, r, w8, row), want_dyp), want_h);
}
MlpBwd mlp8_bwd(const Tensor& dy, const Tensor& r, const Tensor& w8, const ScaledGrad& sg, bool want_h) {
  const Tensor& row = sg.row;
  const int64_t M = check_bwd(dy, r, w8, row), d = last_dim(dy), F = r.size(1);
  MlpBwd o;
  o.dy8 = sg.bytes, o.dyp = sg.padded;
  o.dx = make_rows(dy.sizes(), M, d, dy);
  o.dpre = make({M, F}, BF16, dy);
  if (want_h) o.h = make({M, F}, BF16, dy);
  o.dp8 = make({M, F}, U8, dy);
  TFB_CALL(tfb_mlp8_bwd, ptr(o.dy8), ptr(r), ptr(w8), ptr(row), ptr(o.dx), ptr(o.h), ptr(o.dpre), ptr(o.dp8), M, d, F, stream());
  return o;
}

MlpBwd mlp8_bwd_q(const Tensor& dy, const Tensor& r, const Tensor& w8, const Tensor& row, double limit, bool want_dpre) {
  return mlp8_bwd_q(dy, r, w8, at_scale(dy, row, check_bwd(dy, r, w8, row), false), limit, want_dpre);
}
MlpBwd mlp8_bwd_q(const Tensor& dy, const Tensor& r, const Tensor& w8, const ScaledGrad& sg, double limit, bool want_dpre) {
  const Tensor& row = sg.row;
  const int64_t M = check_bwd(dy, r, w8, row), d = last_dim(dy), F = r.size(1);
  MlpBwd o;
  o.dy8 = sg.bytes;
  o.dx = make_rows(dy.sizes(), M, d, dy);
  if (want_dpre) o.dpre = make({M, F}, BF16, dy);
  o.dp8 = make({M, F}, U8, dy);
  o.hq8 = make({M, F}, U8, dy);
  TFB_CALL(tfb_mlp8_bwd_q, ptr(o.dy8), ptr(r), ptr(w8), ptr(row), ptr(o.dx), nullptr, ptr(o.dpre), ptr(o.dp8), ptr(o.hq8), limit, M, d, F,
           stream());
  return o;
}

bool mlp8_bwd_dw8_applies(const Tensor& r, int64_t d) { return tfb_mlp8_bwd_dw8_applies(r.size(0), d, r.size(1), WORKSPACE_BYTES) == 0; }

Tensor mlp8_bwd_dw8(const Tensor& dy, const Tensor& r, const Tensor& w8, const ScaledGrad& sg, double limit, const Tensor& x8, const Scale& x_scale,
                    const std::function<DwOut()>& outputs) {
  const Tensor &row = sg.row, &dy8 = sg.bytes;
  chk(x8, U8);
  const int64_t M = check_bwd(dy, r, w8, row), d = last_dim(dy), F = r.size(1);
  TORCH_CHECK_VALUE(x8.numel() == M * d && last_dim(x8) == d, "operand shapes");
  const DwOut o = outputs();
  TORCH_CHECK_VALUE(o.fc.numel() == F * d && o.proj.numel() == F * d && o.fc.scalar_type() == o.proj.scalar_type(), "bad outputs");
  const Tensor dx = make_rows(dy.sizes(), M, d, dy), dp8 = make({M, F}, U8, dy), hq8 = make({M, F}, U8, dy);
  TFB_CALL(tfb_mlp8_bwd_dw8, ptr(dy8), ptr(r), ptr(w8), ptr(row), ptr(dx), ptr(dp8), ptr(hq8), limit, ptr(x8), x_scale.imm, ptr(x_scale.dev),
           ptr(o.fc), ptr(o.proj), M, d, F, o.fc.scalar_type() == F32, o.accumulate, WORKSPACE_BYTES, stream());
  return dx;
}

void mlp8_dw8(const Tensor& x8, const Tensor& dp8, const Tensor& hq8, const Tensor& dy8, const Tensor& row, const Scale& x_scale,
              Tensor& dw_fc, Tensor& dw_proj, bool accumulate, at::ScalarType out_dtype) {
  chk(x8, U8), chk(dp8, U8), chk(hq8, U8), chk(dy8, U8), chk(row, F32);
  const int64_t d = last_dim(x8), M = x8.numel() / d, F = dp8.size(1);
  TORCH_CHECK_VALUE(dp8.size(0) == M && hq8.sizes() == dp8.sizes() && dy8.numel() == M * d && dy8.size(-1) == d, "operand shapes");
  TORCH_CHECK_VALUE(dw_fc.defined() == dw_proj.defined(), "give both outputs or neither");
  dw_fc = Out2::get(dw_fc, {F, d}, out_dtype, accumulate, x8);
  dw_proj = Out2::get(dw_proj, {d, F}, out_dtype, accumulate, x8);
  TORCH_CHECK_VALUE(dw_fc.scalar_type() == dw_proj.scalar_type(), "bad outputs");
  const Tensor ws = workspace(x8);
  TFB_CALL(tfb_mlp8_dw8, ptr(x8), ptr(dp8), ptr(hq8), ptr(dy8), ptr(row), x_scale.imm, ptr(dw_fc), ptr(dw_proj), M, d, F,
           dw_fc.scalar_type() == F32, accumulate, ptr(ws), ws.numel() * 4, ptr(x_scale.dev), stream());
}

Tensor mlp_dw_proj(const Tensor& dy, const Tensor& r, Tensor out, bool accumulate, at::ScalarType out_dtype) {
  chk(dy), chk(r);
  const int64_t d = last_dim(dy), M = dy.numel() / d, F = r.size(1);
  check_rows(r, M, F);
  out = Out2::get(out, {d, F}, out_dtype, accumulate, dy);
  const Tensor ws = workspace(dy);
  TFB_CALL(tfb_mlp_dw_proj, ptr(dy), ptr(r), ptr(out), M, d, F, out.scalar_type() == F32, accumulate, ptr(ws), ws.numel() * 4, stream());
  return out;
}

std::tuple<Tensor, Tensor> mlp_fwd(const Tensor& x, const Tensor& w_fc, const Tensor& w_proj) {
  chk(x), chk(w_fc), chk(w_proj);
  const int64_t d = last_dim(x), M = x.numel() / d, F = w_fc.size(0);
  TORCH_CHECK_VALUE(w_fc.sizes() == at::IntArrayRef({F, d}) && w_proj.sizes() == at::IntArrayRef({d, F}), "w_fc is [F, d], w_proj is [d, F]");
  Tensor y = make_like(x), r = make({M, F}, BF16, x), h = make({M, F}, BF16, x);
  TFB_CALL(tfb_mlp_fwd, ptr(x), ptr(w_fc), ptr(w_proj), ptr(y), ptr(r), ptr(h), M, d, F, stream());
  return {y, r};
}

MlpBwd mlp_bwd(const Tensor& dy, const Tensor& r, const Tensor& w_fc, const Tensor& w_proj, bool want_h) {
  chk(dy), chk(r), chk(w_fc), chk(w_proj);
  const int64_t d = last_dim(dy), M = dy.numel() / d, F = w_fc.size(0);
  TORCH_CHECK_VALUE(r.sizes() == at::IntArrayRef({M, F}) && w_fc.sizes() == at::IntArrayRef({F, d}) &&
                        w_proj.sizes() == at::IntArrayRef({d, F}), "shapes differ");
  MlpBwd o;
  o.dx = make_like(dy);
  o.dpre = make({M, F}, BF16, dy);
  if (want_h) o.h = make({M, F}, BF16, dy);
  TFB_CALL(tfb_mlp_bwd, ptr(dy), ptr(r), ptr(w_fc), ptr(w_proj), ptr(o.dx), ptr(o.h), ptr(o.dpre), M, d, F, stream());
  return o;
}

// ----------------------------------------------------------------------------------------------------------- attention
View bhtd(const Tensor& t) {
  TORCH_CHECK(t.dim() == 4 && t.stride(3) == 1, "head dimension must be contiguous");
  return {ptr(t), {t.stride(0), t.stride(1), t.stride(2)}};
}
View bthd(const Tensor& t) {
  TORCH_CHECK(t.dim() == 4 && t.stride(3) == 1, "head dimension must be contiguous");
  return {ptr(t), {t.stride(0), t.stride(2), t.stride(1)}};
}
View third(const Tensor& t, int i, int64_t T, int64_t C, int64_t D, int64_t row) {
  return {static_cast<char*>(ptr(t)) + 2 * i * C, {T * row, D, row}};
}

void attn_fwd(const View& q, const View& k, const View& v, const Tensor& o, const Tensor& lse, int64_t B, int64_t H, int64_t T, int64_t D,
              double scale, int64_t band) {
  const long os[3] = {T * H * D, D, H * D};
  if (band)
    TFB_CALL(tfb_attn_fwd_band, q.p, q.s, k.p, k.s, v.p, v.s, ptr(o), os, ptr(lse), B, H, T, D, scale, band, stream());
  else
    TFB_CALL(tfb_attn_fwd, q.p, q.s, k.p, k.s, v.p, v.s, ptr(o), os, ptr(lse), B, H, T, D, scale, stream());
}

void attn_bwd(const View& q, const View& k, const View& v, const View& o, const View& go, const View& dq, const View& dk,
              const View& dv, const Tensor& lse, const Tensor& cos, const Tensor& sin, int64_t B, int64_t H, int64_t T, int64_t D,
              double scale, int64_t band) {
  chk(cos), chk(sin);
  const Tensor delta = scratch(lse, 2 * B * H * T);
  if (band)
    TFB_CALL(tfb_attn_bwd_band, q.p, q.s, k.p, k.s, v.p, v.s, o.p, o.s, go.p, go.s, dq.p, dq.s, dk.p, dk.s, dv.p, dv.s, ptr(lse),
             ptr(delta), ptr(cos), ptr(sin), B, H, T, D, scale, band, stream());
  else if (cos.defined())
    TFB_CALL(tfb_attn_bwd_rope, q.p, q.s, k.p, k.s, v.p, v.s, o.p, o.s, go.p, go.s, dq.p, dq.s, dk.p, dk.s, dv.p, dv.s, ptr(lse),
             ptr(delta), ptr(cos), ptr(sin), B, H, T, D, scale, stream());
  else
    TFB_CALL(tfb_attn_bwd, q.p, q.s, k.p, k.s, v.p, v.s, o.p, o.s, go.p, go.s, dq.p, dq.s, dk.p, dk.s, dv.p, dv.s, ptr(lse), ptr(delta),
             B, H, T, D, scale, stream());
}

namespace {

struct AttnDims {
  int64_t B, H, T, D;
  at::DimVector shape(bool bthd) const { return bthd ? at::DimVector{B, T, H, D} : at::DimVector{B, H, T, D}; }
};
void check_attn(const Tensor& t) {
  TORCH_CHECK_TYPE(t.is_cuda() && t.scalar_type() == BF16, "attention takes bf16 device tensors");
  TORCH_CHECK_VALUE(t.dim() == 4, "attention tensors are 4-D");
}
AttnDims attn_dims(const Tensor& q, bool bthd) {
  check_attn(q);
  return {q.size(0), q.size(bthd ? 2 : 1), q.size(bthd ? 1 : 2), q.size(3)};
}
// The entry points see only pointers and strides: a tensor of the wrong shape, or a log-sum-exp that is not fp32 [B, H, T] dense,
// would be an out-of-bounds access on the device.
AttnDims check_attn_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& go, const Tensor& lse,
                        const Tensor& dq, const Tensor& dk, const Tensor& dv, bool bthd, bool out_bthd) {
  for (const Tensor* t : {&q, &k, &v, &o, &go, &dq, &dk, &dv}) check_attn(*t);
  const AttnDims m = attn_dims(q, bthd);
  TORCH_CHECK_VALUE(m.T % 128 == 0 && (m.D == 64 || m.D == 128), "attention takes T % 128 == 0 and D 64 or 128");
  TORCH_CHECK_VALUE(k.sizes() == q.sizes() && v.sizes() == q.sizes(), "q, k, v shapes differ");
  for (const Tensor* t : {&o, &go}) TORCH_CHECK_VALUE(t->sizes() == m.shape(true), "o and do are [B, T, H, D]");
  for (const Tensor* t : {&dq, &dk, &dv}) TORCH_CHECK_VALUE(t->sizes() == m.shape(out_bthd), "dq, dk, dv shapes do not match out_layout");
  TORCH_CHECK_VALUE(lse.is_cuda() && lse.scalar_type() == F32 && lse.is_contiguous() && lse.numel() == m.B * m.H * m.T,
                    "lse is fp32 [B, H, T] contiguous");
  return m;
}

}  // namespace

std::tuple<Tensor, Tensor> attention(const Tensor& q, const Tensor& k, const Tensor& v, double scale, bool bthd, int64_t band) {
  const AttnDims m = attn_dims(q, bthd);
  for (const Tensor* t : {&k, &v}) {
    check_attn(*t);
    TORCH_CHECK_VALUE(t->sizes() == q.sizes(), "q, k, v shapes differ");
  }
  Tensor o = make(m.shape(true), BF16, q), lse = make({m.B, m.H, m.T}, F32, q);
  attn_fwd(layout(q, bthd), layout(k, bthd), layout(v, bthd), o, lse, m.B, m.H, m.T, m.D, scale, band);
  return {o, lse};
}

void attention_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& go, const Tensor& lse, double scale,
                   bool bthd_, const Tensor& dq, const Tensor& dk, const Tensor& dv, bool out_bthd, const Tensor& cos, const Tensor& sin,
                   int64_t band) {
  const AttnDims m = check_attn_bwd(q, k, v, o, go, lse, dq, dk, dv, bthd_, out_bthd);
  attn_bwd(layout(q, bthd_), layout(k, bthd_), layout(v, bthd_), bthd(o), bthd(go), layout(dq, out_bthd), layout(dk, out_bthd),
           layout(dv, out_bthd), lse, cos, sin, m.B, m.H, m.T, m.D, scale, band);
}

void attention_bwd_static(const Tensor& q_, const Tensor& k_, const Tensor& v_, const Tensor& o_, const Tensor& go_, const Tensor& lse,
                          double scale, bool bthd_, const Tensor& dq_, const Tensor& dk_, const Tensor& dv_, bool out_bthd) {
  const AttnDims m = check_attn_bwd(q_, k_, v_, o_, go_, lse, dq_, dk_, dv_, bthd_, out_bthd);
  const View q = layout(q_, bthd_), k = layout(k_, bthd_), v = layout(v_, bthd_), o = bthd(o_), go = bthd(go_), dq = layout(dq_, out_bthd),
             dk = layout(dk_, out_bthd), dv = layout(dv_, out_bthd);
  TFB_CALL(tfb_attn_bwd_static, q.p, q.s, k.p, k.s, v.p, v.s, o.p, o.s, go.p, go.s, dq.p, dq.s, dk.p, dk.s, dv.p, dv.s, ptr(lse), m.B, m.H,
           m.T, m.D, scale, stream());
}

RowView row_view(const Tensor& t) {
  TORCH_CHECK_TYPE(t.is_cuda() && t.scalar_type() == BF16 && t.dim() > 0 && t.stride(-1) == 1,
                   "expected a bf16 device tensor with contiguous rows");
  if (t.is_contiguous()) return {t.numel() / last_dim(t), t.size(-1)};
  TORCH_CHECK_VALUE(t.dim() == 2, "a strided operand is a matrix");
  return {t.size(0), t.stride(0)};
}

void rope(const Tensor& x, const Tensor& cos, const Tensor& sin, const Tensor& out, int64_t rows, int64_t T, int64_t nheads, int64_t D,
          int64_t x_stride, int64_t out_stride, bool inverse) {
  chk(cos), chk(sin);
  TFB_CALL(tfb_rope, ptr(x), ptr(cos), ptr(sin), ptr(out), rows, T, nheads, D, x_stride, out_stride, inverse, stream());
}

void rope_norm_fwd(const Tensor& x, const Tensor& cos, const Tensor& sin, const Tensor& r, const Tensor& y, const Tensor& inv,
                   int64_t rows, int64_t T, int64_t nheads, int64_t D, int64_t x_stride, double eps) {
  chk(cos), chk(sin);
  TFB_CALL(tfb_rope_norm_fwd, ptr(x), ptr(cos), ptr(sin), ptr(r), ptr(y), ptr(inv), rows, T, nheads, D, x_stride, nheads * D, nheads * D,
           eps, stream());
}

void rope_norm_bwd(const Tensor& g, const Tensor& r, const Tensor& inv, const Tensor& cos, const Tensor& sin, const Tensor& out,
                   int64_t rows, int64_t T, int64_t nheads, int64_t D, int64_t g_stride, int64_t out_stride) {
  chk(cos), chk(sin), chk(r), chk(inv, F32);
  TFB_CALL(tfb_rope_norm_bwd, ptr(g), ptr(r), ptr(inv), ptr(cos), ptr(sin), ptr(out), rows, T, nheads, D, g_stride, nheads * D, out_stride,
           stream());
}

// --------------------------------------------------------------------------------------- elementwise, embedding, AdamW
Tensor relu2(const Tensor& a, const Tensor& b, int mode) {
  chk(a), chk(b);
  Tensor out = make_like(a);
  TFB_CALL(tfb_relu2, ptr(a), ptr(b), ptr(out), a.numel(), mode, stream());
  return out;
}

static int is64(const Tensor& idx) {
  TORCH_CHECK_TYPE(idx.is_cuda() && (idx.scalar_type() == at::kLong || idx.scalar_type() == I32), "idx must be an int32/int64 device tensor");
  return idx.scalar_type() == at::kLong;
}

Tensor embedding_fwd(const Tensor& idx_, const Tensor& w) {
  chk(w);
  const int i64 = is64(idx_);
  const Tensor idx = dense(idx_);
  const int64_t V = w.size(0), C = w.size(1);
  at::DimVector shape(idx.sizes());
  shape.push_back(C);
  Tensor out = make(shape, BF16, w);
  TFB_CALL(tfb_embedding_fwd, ptr(idx), i64, ptr(w), ptr(out), idx.numel(), C, V, stream());
  return out;
}

void embedding_bwd(const Tensor& idx_, const Tensor& dy, const Tensor& dw) {
  chk(dy), chk(dw, F32);
  const int i64 = is64(idx_);
  const Tensor idx = dense(idx_);
  const int64_t n = idx.numel(), V = dw.size(0);
  const Tensor scr = make({tfb_embedding_bwd_scratch_ints(n, V)}, I32, dw);
  TFB_CALL(tfb_embedding_bwd_grouped, ptr(idx), i64, ptr(dy), ptr(dw), n, dy.size(-1), V, ptr(scr), stream());
}

void fill_f32(const Tensor& t, double v) {
  chk(t, F32);
  TFB_CALL(tfb_fill_f32, ptr(t), v, t.numel(), stream());
}

void adamw(const Tensor& p, const Tensor& g, const Tensor& m, const Tensor& v, double step, double lr, double beta1, double beta2,
           double eps, double weight_decay, const Tensor& p_bf16) {
  chk(p, F32), chk(m, F32), chk(v, F32), chk(g, g.scalar_type()), chk(p_bf16);
  TORCH_CHECK_TYPE(g.scalar_type() == F32 || g.scalar_type() == BF16, "grad must be fp32 or bf16");
  TFB_CALL(tfb_adamw, ptr(p), ptr(g), g.scalar_type() == F32, ptr(m), ptr(v), ptr(p_bf16), p.numel(), lr, weight_decay, 1.0 - beta1,
           1.0 - beta2, eps, 1.0 - std::pow(beta1, step), 1.0 - std::pow(beta2, step), stream());
}

// ----------------------------------------------------------------------------------------------------------- loss head
Tensor targets_of(const Tensor& t) {
  TORCH_CHECK_TYPE(t.is_cuda() && (t.scalar_type() == at::kLong || t.scalar_type() == I32), "targets must be an int32/int64 device tensor");
  return dense(t);
}

Tensor loss_row_weights(const Tensor& tg, bool mean, int64_t V) {
  Tensor w = scratch(tg, tg.numel());
  TFB_CALL(tfb_loss_row_weights, ptr(tg), is64(tg), ptr(w), tg.numel(), mean, V, stream());
  return w;
}

std::tuple<Tensor, Tensor> loss_fwd(const Tensor& logits, const Tensor& tg, const Tensor& row_w, double softcap, int64_t N, int64_t V) {
  chk(logits), chk(row_w, F32);
  Tensor loss = scratch(logits, N), lse = scratch(logits, N);
  TFB_CALL(tfb_loss_fwd, ptr(logits), ptr(tg), is64(tg), ptr(row_w), ptr(loss), ptr(lse), N, V, softcap, stream());
  return {loss, lse};
}

std::tuple<Tensor, Tensor> loss_fwd_bwd(const Tensor& logits, const Tensor& tg, const Tensor& row_w, double softcap, int64_t N, int64_t V) {
  chk(logits), chk(row_w, F32);
  Tensor loss = scratch(logits, N), lse = scratch(logits, N);
  TFB_CALL(tfb_loss_fwd_bwd, ptr(logits), ptr(tg), is64(tg), ptr(row_w), ptr(loss), ptr(lse), N, V, softcap, stream());
  return {loss, lse};
}

void loss_bwd(const Tensor& logits, const Tensor& tg, const Tensor& lse, const Tensor& grow, const Tensor& out, double softcap, int64_t N,
              int64_t V) {
  chk(logits), chk(lse, F32), chk(grow, F32);
  TFB_CALL(tfb_loss_bwd, ptr(logits), ptr(tg), is64(tg), ptr(lse), ptr(grow), ptr(out), N, V, softcap, stream());
}

std::tuple<Tensor, Tensor, Tensor> lmhead_fwd(const Tensor& x, const Tensor& W, const Tensor& tg, double softcap, const Tensor& row_w) {
  chk(x), chk(W), chk(row_w, F32);
  const int64_t d = last_dim(x), N = x.numel() / d, V = W.size(0);
  Tensor logits = make({N, V}, BF16, x), part = scratch(x, N * (V / 64) * 2), loss = scratch(x, N), lse = scratch(x, N);
  TFB_CALL(tfb_lmhead_fwd, ptr(x), ptr(W), ptr(tg), is64(tg), ptr(row_w), ptr(logits), ptr(part), ptr(loss), ptr(lse), N, d, V, softcap,
           stream());
  return {logits, loss, lse};
}

// -------------------------------------------------------------------------------------------------- mixture of experts
MoeRoute moe_route(const Tensor& h, const Tensor& wr, int64_t topk, const Tensor& bias, bool want_logits) {
  chk(h), chk(wr, F32), chk(bias, F32);
  const int64_t d = last_dim(h), N = h.numel() / d, E = wr.size(0);
  MoeRoute o{make({N, E}, F32, h), make({N, topk}, I32, h), make({N, topk}, F32, h), want_logits ? make({N, E}, F32, h) : Tensor()};
  TFB_CALL(tfb_moe_route, ptr(h), ptr(wr), ptr(bias), ptr(o.logits), ptr(o.p), ptr(o.idx), ptr(o.gate), N, d, E, topk, stream());
  return o;
}

MoeTab moe_tables(const Tensor& idx, int64_t E, int64_t seq_len, int64_t capacity) {
  chk(idx, I32);
  const int64_t N = idx.size(0), topk = idx.size(1), nw = (N + 63) / 64;
  MoeTab t;
  t.rmax = tfb_moe_max_rows(N, E, topk);
  t.cnt = make({E}, I32, idx), t.seg = make({E + 1}, I32, idx), t.tile_expert = make({t.rmax / 128}, I32, idx);
  t.slot = make({N, topk}, I32, idx), t.tok = make({t.rmax}, I32, idx), t.ksel = make({t.rmax}, I32, idx);
  t.capped = capacity >= 0, t.capacity = capacity;
  if (!t.capped) {
    const Tensor scr = make({nw * E}, I32, idx);
    TFB_CALL(tfb_moe_tables, ptr(idx), ptr(t.cnt), ptr(t.seg), ptr(t.tile_expert), ptr(t.slot), ptr(t.tok), ptr(t.ksel), ptr(scr), N, E, topk,
             t.rmax, stream());
    return t;
  }
  TORCH_CHECK_VALUE(seq_len >= 0, "a capacity is counted per sequence: seq_len is needed");
  t.cnt_all = make({E}, I32, idx);
  const Tensor scr = make({2 * nw * E}, I32, idx);
  TFB_CALL(tfb_moe_tables_cap, ptr(idx), ptr(t.cnt), ptr(t.cnt_all), ptr(t.seg), ptr(t.tile_expert), ptr(t.slot), ptr(t.tok), ptr(t.ksel),
           ptr(scr), N, seq_len, capacity, E, topk, t.rmax, stream());
  return t;
}

std::tuple<Tensor, Tensor> moe_gather(const Tensor& h, const MoeTab& tab, const Scale* x_scale, bool want_xs) {
  chk(h);
  const int64_t d = last_dim(h);
  Tensor xs, xs8;
  if (want_xs || !x_scale) xs = make({tab.rmax, d}, BF16, h);
  if (x_scale) xs8 = make({tab.rmax, d}, U8, h);
  TFB_CALL(tfb_moe_gather, ptr(h), ptr(tab.tok), x_scale ? ptr(x_scale->dev) : nullptr, x_scale ? x_scale->imm : 1.0, ptr(xs), ptr(xs8),
           tab.rmax, d, stream());
  return {xs, xs8};
}

std::tuple<Tensor, Tensor> moe_mlp8_fwd(const Tensor& xs8, const Tensor& w8, const Tensor& rows, const MoeTab& tab, int64_t F) {
  chk(xs8, U8), chk(w8, U8), chk(rows, F32);
  const int64_t rmax = xs8.size(0), d = xs8.size(1);
  Tensor ys = make({rmax, d}, BF16, xs8), r = make({rmax, F}, BF16, xs8), h8 = make({rmax, F}, U8, xs8);
  TFB_CALL(tfb_moe_mlp8_fwd, ptr(xs8), ptr(w8), ptr(rows), ptr(tab.tile_expert), ptr(ys), ptr(r), ptr(h8), rmax, d, F, stream());
  return {ys, r};
}

std::tuple<Tensor, Tensor, Tensor> moe_mlp_fwd(const Tensor& xs, const Tensor& w_fc, const Tensor& w_proj, const MoeTab& tab) {
  chk(xs), chk(w_fc), chk(w_proj);
  const int64_t rmax = xs.size(0), d = xs.size(1), E = w_fc.size(0), F = w_fc.size(1);
  TORCH_CHECK_VALUE(w_fc.sizes() == at::IntArrayRef({E, F, d}) && w_proj.sizes() == at::IntArrayRef({E, d, F}),
                    "moe_mlp_fwd: w_fc [E,F,d] and w_proj [E,d,F] expected");
  Tensor ys = make({rmax, d}, BF16, xs), r = make({rmax, F}, BF16, xs), h = make({rmax, F}, BF16, xs);
  TFB_CALL(tfb_moe_mlp_fwd, ptr(xs), ptr(w_fc), ptr(w_proj), ptr(tab.tile_expert), ptr(ys), ptr(r), ptr(h), rmax, d, F, stream());
  return {ys, r, h};
}

Tensor moe_combine(const Tensor& ys, const MoeTab& tab, const Tensor& gate, at::IntArrayRef out_shape) {
  chk(ys), chk(gate, F32);
  Tensor out = make(out_shape, BF16, ys);
  TFB_CALL(tfb_moe_combine, ptr(ys), ptr(tab.slot), ptr(gate), ptr(out), gate.size(0), ys.size(1), gate.size(1), stream());
  return out;
}

CombineGrad moe_combine_bwd(const Tensor& dout, const Tensor& ys, const MoeTab& tab, const Tensor& gate, bool want_rowmax, bool want_dys) {
  chk(dout), chk(ys), chk(gate, F32);
  const int64_t rmax = ys.size(0), d = ys.size(1);
  CombineGrad o{want_dys ? make_like(ys) : Tensor(), make_like(gate), {}};
  // the kernel writes the gate gradient of every assignment that holds a row; a skipped one's is zero
  if (tab.capped) fill_f32(o.dgate, 0.0);
  if (want_rowmax) {
    o.rowmax = scratch(ys, rmax);
    TFB_CALL(tfb_moe_combine_bwd_rowmax, ptr(dout), ptr(ys), ptr(tab.tok), ptr(tab.ksel), ptr(gate), ptr(o.dys), ptr(o.dgate), ptr(o.rowmax),
             rmax, d, gate.size(1), stream());
  } else {
    TFB_CALL(tfb_moe_combine_bwd, ptr(dout), ptr(ys), ptr(tab.tok), ptr(tab.ksel), ptr(gate), ptr(o.dys), ptr(o.dgate), rmax, d, gate.size(1),
             stream());
  }
  return o;
}

Tensor moe_backward_scales_rowmax(const Tensor& rowmax, const Tensor& rows, const MoeTab& tab, int64_t d) {
  chk(rowmax, F32), chk(rows, F32);
  Tensor out = make_like(rows);
  TFB_CALL(tfb_moe_backward_scales_rowmax, ptr(rowmax), ptr(tab.seg), ptr(rows), ptr(out), d, rows.size(0), stream());
  return out;
}

Tensor moe_quant(const Tensor& x, const Tensor& rows, int64_t col, int64_t fmt, const MoeTab& tab) {
  chk(x), chk(rows, F32);
  Tensor out = make(x.sizes(), U8, x);
  TFB_CALL(tfb_moe_quant, ptr(x), ptr(tab.tile_expert), ptr(rows), col, fmt, ptr(out), x.size(0), x.size(1), stream());
  return out;
}

Tensor moe_quant_dout(const Tensor& dout, const Tensor& gate, const Tensor& rows, const MoeTab& tab) {
  chk(dout), chk(gate, F32), chk(rows, F32);
  const int64_t d = last_dim(dout);
  Tensor out = make({tab.rmax, d}, U8, dout);
  TFB_CALL(tfb_moe_quant_dout, ptr(dout), ptr(tab.tok), ptr(tab.ksel), ptr(gate), ptr(tab.tile_expert), ptr(rows), 5, ptr(out), tab.rmax, d,
           gate.size(1), stream());
  return out;
}

MlpBwd moe_mlp8_bwd(const Tensor& dys, const Tensor& r, const Tensor& w8, const Tensor& rows, const MoeTab& tab) {
  chk(dys), chk(r), chk(w8, U8);
  const int64_t rmax = dys.size(0), d = dys.size(1), F = r.size(1);
  MlpBwd o;
  o.dy8 = moe_quant(dys, rows, 5, E5M2, tab);
  o.dx = make({rmax, d}, BF16, dys), o.dpre = make({rmax, F}, BF16, dys), o.dp8 = make({rmax, F}, U8, dys);
  TFB_CALL(tfb_moe_mlp8_bwd, ptr(o.dy8), ptr(r), ptr(w8), ptr(rows), ptr(tab.tile_expert), ptr(o.dx), ptr(o.dpre), ptr(o.dp8), rmax, d, F,
           stream());
  return o;
}

MlpBwd moe_mlp8_bwd_q(const Tensor& dy8, const Tensor& r, const Tensor& w8, const Tensor& rows, const MoeTab& tab, double limit) {
  chk(dy8, U8), chk(r), chk(w8, U8);
  const int64_t rmax = dy8.size(0), d = dy8.size(1), F = r.size(1);
  MlpBwd o;
  o.dy8 = dy8;
  o.dx = make({rmax, d}, BF16, r), o.dp8 = make({rmax, F}, U8, r), o.hq8 = make({rmax, F}, U8, r);
  TFB_CALL(tfb_moe_mlp8_bwd_q, ptr(o.dy8), ptr(r), ptr(w8), ptr(rows), ptr(tab.tile_expert), ptr(o.dx), nullptr, ptr(o.dp8), ptr(o.hq8), limit,
           rmax, d, F, stream());
  return o;
}

MlpBwd moe_mlp_bwd(const Tensor& dys, const Tensor& r, const Tensor& w_fc, const Tensor& w_proj, const MoeTab& tab) {
  chk(dys), chk(r), chk(w_fc), chk(w_proj);
  const int64_t rmax = dys.size(0), d = dys.size(1), F = r.size(1);
  MlpBwd o;
  o.dx = make({rmax, d}, BF16, dys), o.dpre = make({rmax, F}, BF16, dys);
  TFB_CALL(tfb_moe_mlp_bwd, ptr(dys), ptr(r), ptr(w_fc), ptr(w_proj), ptr(tab.tile_expert), ptr(o.dx), ptr(o.dpre), rmax, d, F, stream());
  return o;
}

static void moe_dw_outputs(Tensor& dw_fc, Tensor& dw_proj, int64_t E, int64_t F, int64_t d, bool accumulate, at::ScalarType out_dtype,
                           const Tensor& like) {
  TORCH_CHECK_VALUE(dw_fc.defined() == dw_proj.defined(), "give both outputs or neither");
  dw_fc = Out2::get(dw_fc, {E, F, d}, out_dtype, accumulate, like);
  dw_proj = Out2::get(dw_proj, {E, d, F}, out_dtype, accumulate, like);
  TORCH_CHECK_VALUE(dw_fc.scalar_type() == dw_proj.scalar_type(), "bad outputs");
}

void moe_dw8(const Tensor& xs8, const Tensor& dp8, const Tensor& hq8, const Tensor& dy8, const Tensor& rows, double x_scale,
             const MoeTab& tab, Tensor& dw_fc, Tensor& dw_proj, int64_t E, bool accumulate, at::ScalarType out_dtype) {
  chk(xs8, U8), chk(dp8, U8), chk(hq8, U8), chk(dy8, U8), chk(rows, F32);
  const int64_t d = xs8.size(1), F = dp8.size(1);
  moe_dw_outputs(dw_fc, dw_proj, E, F, d, accumulate, out_dtype, xs8);
  TFB_CALL(tfb_moe_dw8_rows, ptr(xs8), ptr(dp8), ptr(hq8), ptr(dy8), ptr(rows), x_scale, ptr(tab.seg), ptr(dw_fc), ptr(dw_proj), E, d, F,
           dw_fc.scalar_type() == F32, accumulate, xs8.size(0), stream());
}

void moe_dw(const Tensor& dpre, const Tensor& xs, const Tensor& dys, const Tensor& r, const MoeTab& tab, Tensor& dw_fc, Tensor& dw_proj,
            int64_t E, bool accumulate, at::ScalarType out_dtype) {
  const int64_t d = xs.size(1), F = r.size(1);
  chk(dpre), chk(xs), chk(dys), chk(r);
  moe_dw_outputs(dw_fc, dw_proj, E, F, d, accumulate, out_dtype, xs);
  TFB_CALL(tfb_moe_dw, ptr(dpre), ptr(xs), ptr(dys), ptr(r), ptr(tab.seg), ptr(dw_fc), ptr(dw_proj), E, d, F, dw_fc.scalar_type() == F32,
           accumulate, stream());
}

std::tuple<Tensor, Tensor> moe_aux_fwd(const Tensor& p, const Tensor& logits, const MoeTab& tab, int64_t topk) {
  chk(p, F32), chk(logits, F32);
  const int64_t N = p.size(0), E = p.size(1);
  Tensor terms = scratch(p, 2 + E), lse = scratch(p, N), scr = scratch(p, 64 * 17);
  TFB_CALL(tfb_moe_aux_fwd, ptr(p), ptr(logits), ptr(tab.capped ? tab.cnt_all : tab.cnt), ptr(terms), ptr(lse), ptr(scr), N, E, topk,
           stream());
  return {terms, lse};
}

std::tuple<Tensor, Tensor> moe_aux_seq_fwd(const Tensor& p, const Tensor& idx, int64_t T, int64_t topk) {
  chk(p, F32), chk(idx, I32);
  const int64_t N = p.size(0), E = p.size(1);
  TORCH_CHECK_VALUE(T > 0 && N % T == 0, "moe_aux_seq_fwd: ", N, " tokens are not whole sequences of ", T);
  Tensor fs = make({N / T, E}, F32, p), term = scratch(p, 1), scr = scratch(p, N / T);
  TFB_CALL(tfb_moe_aux_seq_fwd, ptr(p), ptr(idx), ptr(fs), ptr(term), ptr(scr), N, T, E, topk, stream());
  return {term, fs};
}

RouteGrad moe_route_bwd(const Tensor& dgate, const Tensor& p, const Tensor& idx, const Tensor& dxs, const MoeTab& tab, const Tensor& h,
                        const Tensor& wr, Tensor dwr, bool accumulate, const MoeAux* aux) {
  const int64_t d = last_dim(h), N = h.numel() / d, E = wr.size(0), topk = idx.size(1);
  if (!dwr.defined()) {
    dwr = make({E, d}, F32, h);
    accumulate = false;
  }
  RouteGrad o{make_like(h), dwr, make({N, E}, F32, h)};
  const Tensor scr = scratch(h, 64 * E * d);
  if (!aux) {
    TFB_CALL(tfb_moe_route_bwd, ptr(dgate), ptr(p), ptr(idx), ptr(dxs), ptr(tab.slot), ptr(h), ptr(wr), ptr(o.dlogits), ptr(o.dh), ptr(dwr),
             accumulate, ptr(scr), N, d, E, topk, stream());
    return o;
  }
  chk(aux->terms, F32), chk(aux->lse, F32), chk(aux->gaux, F32), chk(aux->fs, F32);
  if (aux->fs.defined()) {
    TORCH_CHECK_VALUE(N % aux->seq_len == 0 && aux->fs.sizes() == at::IntArrayRef({N / aux->seq_len, E}),
                      "moe_route_bwd: fs must be [N / seq_len, E]");
    TFB_CALL(tfb_moe_route_bwd_aux_seq, ptr(dgate), ptr(p), ptr(idx), ptr(dxs), ptr(tab.slot), ptr(h), ptr(wr), ptr(o.dlogits), ptr(o.dh),
             ptr(dwr), accumulate, ptr(scr), ptr(aux->terms), ptr(aux->lse), ptr(aux->gaux), aux->alpha, aux->beta, ptr(aux->fs), aux->gamma,
             aux->seq_len, N, d, E, topk, stream());
  } else {
    TFB_CALL(tfb_moe_route_bwd_aux, ptr(dgate), ptr(p), ptr(idx), ptr(dxs), ptr(tab.slot), ptr(h), ptr(wr), ptr(o.dlogits), ptr(o.dh),
             ptr(dwr), accumulate, ptr(scr), ptr(aux->terms), ptr(aux->lse), ptr(aux->gaux), aux->alpha, aux->beta, N, d, E, topk, stream());
  }
  return o;
}

}  // namespace tfb
