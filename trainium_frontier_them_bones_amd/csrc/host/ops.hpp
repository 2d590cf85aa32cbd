// The entry points on tensors: checks, outputs and scratch from torch's allocator, one library call (or a short fixed
// sequence) on the current stream. No autograd here. An undefined Tensor stands for "not given".
#pragma once
#include <functional>

#include "common.hpp"

namespace tfb {

// GEMM. The explicit sizes let the callers hand over tensors of any leading shape.
void gemm(const Tensor& a, const Tensor& b, const Tensor& out, int64_t M, int64_t N, int64_t K, bool ta, bool tb, bool accumulate,
          const Tensor& alpha = {});
// dx = gy w and dw (+)= gy^T x in one launch, where linear_bwd_applies; bf16 operands, checked by the caller
bool linear_bwd_applies(int64_t M, int64_t N, int64_t K);
void linear_bwd(const Tensor& gy, const Tensor& x, const Tensor& w, const Tensor& dx, const Tensor& dw, int64_t M, int64_t N, int64_t K,
                bool accumulate);
Tensor matmul(const Tensor& a, const Tensor& b, bool ta, bool tb, Tensor out, bool accumulate, at::ScalarType out_dtype,
              const Tensor& alpha);
Tensor matmul_res(const Tensor& a, const Tensor& b, const Tensor& res, bool tb);
Tensor qkv_rope(const Tensor& x2, const Tensor& w, const Tensor& cos, const Tensor& sin, int64_t T, int64_t rot_cols, int64_t D = 64);
Tensor workspace(const Tensor& like);   // fp32 split-K scratch of the current stream

// norms
struct NormOut { Tensor s, y, inv, y8; };
NormOut rmsnorm_fwd(const Tensor& x, const Tensor& w, double eps, const Tensor& res);
// rows_out: the rows of y and y8 (0: x's); those beyond x's are zeros
NormOut rmsnorm_fwd_q(const Tensor& x, const Tensor& w, double eps, const Tensor& res, double y8_scale, bool want_y, int64_t rows_out = 0);
struct NormGrad { Tensor dx, dw, amax; };
NormGrad rmsnorm_bwd(const Tensor& gy, const Tensor& s, const Tensor& inv, const Tensor& w, const Tensor& gs, const Tensor& dw,
                     bool accumulate, const Tensor& part, bool want_amax);
std::tuple<Tensor, Tensor, Tensor> block_head_fwd(const Tensor& x, const Tensor& x0, const Tensor& gains, const Tensor& skip, double eps);
struct HeadGrad { Tensor dx, dx0, dskip, dgains; };
HeadGrad block_head_bwd(const Tensor& g_new, const Tensor& g_norm, const Tensor& x, const Tensor& x0, const Tensor& x_new,
                        const Tensor& inv, const Tensor& gains, const Tensor& skip);
std::tuple<Tensor, Tensor, Tensor> mix_tail_fwd(const Tensor& x, const Tensor& lam, int64_t T, double eps);
std::tuple<Tensor, Tensor> mix_tail_bwd(const Tensor& s1, const Tensor& inv, const Tensor& x, const Tensor& lam, int64_t T,
                                        const Tensor& gy, const Tensor& ge);

// fp8 MLP. A scale is a float or a one-element fp32 device tensor.
struct Scale {
  double imm = 0;
  Tensor dev;
  double host() const { return dev.defined() ? dev.item<double>() : imm; }   // (reads the device value back)
};
Tensor mlp8_backward_scales(const Tensor& dy, const Tensor& row, const Tensor& amax_part);
// The scale row and dy's bytes at its scale, whole tiles of rows; padded: dy in bf16 of as many, where it is asked for
struct ScaledGrad {
  Tensor row, bytes, padded;
};
ScaledGrad mlp8_scaled_grad(const Tensor& dy, const Tensor& row, const Tensor& amax_part, bool want_padded);
Tensor amax_scale(const Tensor& x, double limit, int64_t e_lo, int64_t e_hi);
Tensor quant_fp8(const Tensor& x, const void* scale_dev, double scale_imm, int fmt);
Tensor quant_fp8(const Tensor& x, const Scale& s, int fmt);
Tensor gemm_fp8(const Tensor& a8, const Tensor& b8, int fmt_a, const void* dq_a, const void* dq_b, double dq, const Tensor& res,
                at::IntArrayRef out_shape);
Tensor gemm_fp8_tn(const Tensor& g8, const Tensor& a8, int fmt_g, int fmt_a, const void* s_g, const void* s_a, double imm, Tensor out,
                   bool accumulate, at::ScalarType out_dtype);
// The fp8 MLP's calls take any number of rows; r and the byte operands have tile_rows(rows) rows, those beyond the given ones
// from zeros. xp / dyp: x / dy with as many rows (themselves where nothing is to be padded), asked for by want_xp / want_dyp.
inline int64_t tile_rows(int64_t rows) { return (rows + 127) / 128 * 128; }
struct MlpFwd { Tensor y, r, x8, xp; };
MlpFwd mlp8_fwd(const Tensor& x, const Tensor& w8, const Tensor& row, int64_t F, const Scale& x_scale, const Tensor& x8, const Tensor& res,
                bool want_xp = false);
struct MlpBwd { Tensor dx, h, dpre, dp8, hq8, dy8, dyp; };
MlpBwd mlp8_bwd(const Tensor& dy, const Tensor& r, const Tensor& w8, const Tensor& row, bool want_h, bool want_dyp = false);
MlpBwd mlp8_bwd(const Tensor& dy, const Tensor& r, const Tensor& w8, const ScaledGrad& sg, bool want_h);
MlpBwd mlp8_bwd_q(const Tensor& dy, const Tensor& r, const Tensor& w8, const Tensor& row, double limit, bool want_dpre);
MlpBwd mlp8_bwd_q(const Tensor& dy, const Tensor& r, const Tensor& w8, const ScaledGrad& sg, double limit, bool want_dpre);
// dx and both weight gradients at once, where mlp8_bwd_dw8_applies; outputs() is asked for the latter once the operands are checked
struct DwOut {
  Tensor fc, proj;
  bool accumulate;
};
bool mlp8_bwd_dw8_applies(const Tensor& r, int64_t d);
Tensor mlp8_bwd_dw8(const Tensor& dy, const Tensor& r, const Tensor& w8, const ScaledGrad& sg, double limit, const Tensor& x8, const Scale& x_scale,
                    const std::function<DwOut()>& outputs);
void mlp8_dw8(const Tensor& x8, const Tensor& dp8, const Tensor& hq8, const Tensor& dy8, const Tensor& row, const Scale& x_scale,
              Tensor& dw_fc, Tensor& dw_proj, bool accumulate, at::ScalarType out_dtype);
Tensor mlp_dw_proj(const Tensor& dy, const Tensor& r, Tensor out, bool accumulate, at::ScalarType out_dtype);
std::tuple<Tensor, Tensor> mlp_fwd(const Tensor& x, const Tensor& w_fc, const Tensor& w_proj);
MlpBwd mlp_bwd(const Tensor& dy, const Tensor& r, const Tensor& w_fc, const Tensor& w_proj, bool want_h);

// attention: a [.., D] operand through its (batch, head, token) element strides
struct View {
  void* p;
  long s[3];
};
View bhtd(const Tensor& t);                                      // a 4-D tensor [B, H, T, D]
View bthd(const Tensor& t);                                      // a 4-D tensor [B, T, H, D]
inline View layout(const Tensor& t, bool bthd_) { return bthd_ ? bthd(t) : bhtd(t); }
View third(const Tensor& t, int i, int64_t T, int64_t C, int64_t D, int64_t row);   // columns i C .. of a [B T, row] tensor, heads of D
void attn_fwd(const View& q, const View& k, const View& v, const Tensor& o, const Tensor& lse, int64_t B, int64_t H, int64_t T, int64_t D,
              double scale, int64_t band);
void attn_bwd(const View& q, const View& k, const View& v, const View& o, const View& go, const View& dq, const View& dk,
              const View& dv, const Tensor& lse, const Tensor& cos, const Tensor& sin, int64_t B, int64_t H, int64_t T, int64_t D,
              double scale, int64_t band);
// on 4-D tensors [B, H, T, D] or [B, T, H, D], a flag for q, k, v and one for dq, dk, dv
std::tuple<Tensor, Tensor> attention(const Tensor& q, const Tensor& k, const Tensor& v, double scale, bool bthd, int64_t band);
void attention_bwd(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& go, const Tensor& lse, double scale,
                   bool bthd, const Tensor& dq, const Tensor& dk, const Tensor& dv, bool out_bthd, const Tensor& cos, const Tensor& sin,
                   int64_t band);
void attention_bwd_static(const Tensor& q, const Tensor& k, const Tensor& v, const Tensor& o, const Tensor& go, const Tensor& lse,
                          double scale, bool bthd, const Tensor& dq, const Tensor& dk, const Tensor& dv, bool out_bthd);
inline View whole(const Tensor& t, int64_t T, int64_t H, int64_t D) { return {ptr(t), {T * H * D, D, H * D}}; }   // dense [B, T, H, D]
// a 2-D view with contiguous rows, or a dense tensor as rows of its last dimension
struct RowView {
  int64_t rows, stride;
};
RowView row_view(const Tensor& t);
void rope(const Tensor& x, const Tensor& cos, const Tensor& sin, const Tensor& out, int64_t rows, int64_t T, int64_t nheads, int64_t D,
          int64_t x_stride, int64_t out_stride, bool inverse);
void rope_norm_fwd(const Tensor& x, const Tensor& cos, const Tensor& sin, const Tensor& r, const Tensor& y, const Tensor& inv,
                   int64_t rows, int64_t T, int64_t nheads, int64_t D, int64_t x_stride, double eps);
void rope_norm_bwd(const Tensor& g, const Tensor& r, const Tensor& inv, const Tensor& cos, const Tensor& sin, const Tensor& out,
                   int64_t rows, int64_t T, int64_t nheads, int64_t D, int64_t g_stride, int64_t out_stride);

// elementwise, embedding, optimizer
Tensor relu2(const Tensor& a, const Tensor& b, int mode);
Tensor embedding_fwd(const Tensor& idx, const Tensor& w);
void embedding_bwd(const Tensor& idx, const Tensor& dy, const Tensor& dw);
void fill_f32(const Tensor& t, double v);
void adamw(const Tensor& p, const Tensor& g, const Tensor& m, const Tensor& v, double step, double lr, double beta1, double beta2,
           double eps, double weight_decay, const Tensor& p_bf16);

// loss head
Tensor targets_of(const Tensor& t);   // checked and contiguous
Tensor loss_row_weights(const Tensor& tg, bool mean, int64_t V);
std::tuple<Tensor, Tensor> loss_fwd(const Tensor& logits, const Tensor& tg, const Tensor& row_w, double softcap, int64_t N, int64_t V);
std::tuple<Tensor, Tensor> loss_fwd_bwd(const Tensor& logits, const Tensor& tg, const Tensor& row_w, double softcap, int64_t N, int64_t V);
void loss_bwd(const Tensor& logits, const Tensor& tg, const Tensor& lse, const Tensor& grow, const Tensor& out, double softcap, int64_t N,
              int64_t V);
std::tuple<Tensor, Tensor, Tensor> lmhead_fwd(const Tensor& x, const Tensor& W, const Tensor& tg, double softcap, const Tensor& row_w);

// mixture of experts
struct MoeTab {
  Tensor cnt, seg, tile_expert, slot, tok, ksel, cnt_all;
  int64_t rmax = 0, capacity = 0;
  bool capped = false;
};
struct MoeRoute { Tensor p, idx, gate, logits; };
MoeRoute moe_route(const Tensor& h, const Tensor& wr, int64_t topk, const Tensor& bias, bool want_logits);
MoeTab moe_tables(const Tensor& idx, int64_t E, int64_t seq_len, int64_t capacity);   // capacity < 0: dropless
std::tuple<Tensor, Tensor> moe_gather(const Tensor& h, const MoeTab& tab, const Scale* x_scale, bool want_xs);
std::tuple<Tensor, Tensor> moe_mlp8_fwd(const Tensor& xs8, const Tensor& w8, const Tensor& rows, const MoeTab& tab, int64_t F);
std::tuple<Tensor, Tensor, Tensor> moe_mlp_fwd(const Tensor& xs, const Tensor& w_fc, const Tensor& w_proj, const MoeTab& tab);
Tensor moe_combine(const Tensor& ys, const MoeTab& tab, const Tensor& gate, at::IntArrayRef out_shape);
struct CombineGrad { Tensor dys, dgate, rowmax; };
// want_dys false (with want_rowmax): dys is left out, moe_quant_dout makes its bytes
CombineGrad moe_combine_bwd(const Tensor& dout, const Tensor& ys, const MoeTab& tab, const Tensor& gate, bool want_rowmax, bool want_dys = true);
Tensor moe_quant(const Tensor& x, const Tensor& rows, int64_t col, int64_t fmt, const MoeTab& tab);
Tensor moe_quant_dout(const Tensor& dout, const Tensor& gate, const Tensor& rows, const MoeTab& tab);
Tensor moe_backward_scales_rowmax(const Tensor& rowmax, const Tensor& rows, const MoeTab& tab, int64_t d);
MlpBwd moe_mlp8_bwd(const Tensor& dys, const Tensor& r, const Tensor& w8, const Tensor& rows, const MoeTab& tab);
MlpBwd moe_mlp8_bwd_q(const Tensor& dy8, const Tensor& r, const Tensor& w8, const Tensor& rows, const MoeTab& tab, double limit);
MlpBwd moe_mlp_bwd(const Tensor& dys, const Tensor& r, const Tensor& w_fc, const Tensor& w_proj, const MoeTab& tab);
void moe_dw8(const Tensor& xs8, const Tensor& dp8, const Tensor& hq8, const Tensor& dy8, const Tensor& rows, double x_scale,
             const MoeTab& tab, Tensor& dw_fc, Tensor& dw_proj, int64_t E, bool accumulate, at::ScalarType out_dtype);
void moe_dw(const Tensor& dpre, const Tensor& xs, const Tensor& dys, const Tensor& r, const MoeTab& tab, Tensor& dw_fc, Tensor& dw_proj,
            int64_t E, bool accumulate, at::ScalarType out_dtype);
struct MoeAux {
  Tensor terms, lse, gaux, fs;
  double alpha = 0, beta = 0, gamma = 0;
  int64_t seq_len = 0;
};
std::tuple<Tensor, Tensor> moe_aux_fwd(const Tensor& p, const Tensor& logits, const MoeTab& tab, int64_t topk);
std::tuple<Tensor, Tensor> moe_aux_seq_fwd(const Tensor& p, const Tensor& idx, int64_t seq_len, int64_t topk);
struct RouteGrad { Tensor dh, dwr, dlogits; };
RouteGrad moe_route_bwd(const Tensor& dgate, const Tensor& p, const Tensor& idx, const Tensor& dxs, const MoeTab& tab, const Tensor& h,
                        const Tensor& wr, Tensor dwr, bool accumulate, const MoeAux* aux);

}  // namespace tfb
