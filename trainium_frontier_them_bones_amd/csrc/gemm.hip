// bf16 GEMM primitive behind the C-ABI: C[M,N] = op(A) @ op(B), fp32 accumulation, one
// rounding to bf16 (or fp32 output), optional accumulate into C (the in-place weight-gradient
// sum) and split-K through an fp32 workspace for small outputs with a long contraction.
// Replaces the reference's nki_matmul(a, b, trans_a, trans_b) (round1/source/train.py:1137)
// and the torch matmuls its Linear glue issues (round1/source/train.py:8419-8711).
#include "gemm_pp.hpp"
#include "gemm_ring.hpp"

namespace {

template <int LAYP, int LAYQ>
int run(GemmOperand P, GemmOperand Q, int N, int M, int K, void* C, int out_f32, int accumulate, float* ws, long ws_bytes,
        const float* alpha, hipStream_t stream) {
  using Cfg = GemmCfg<128, 128, 2, 2, 2, LAYP, LAYQ>;
  // Long contractions (at least 128 k-tiles) in any operand layout: the persistent 256 x 256 kernel, partial tiles through
  // the fp32 workspace. With 64 or more output tiles the k range is cut into the fewest parts that fill whole rounds of
  // the CUs to 90 % (the LM head's two gradient GEMMs: 384 tiles x 2 = 3 per CU). With fewer (the layers' weight
  // gradients: 9 to 27 tiles of 512 k-tiles) every workgroup gets one work item: as many k ranges per XCD as its 32 CUs
  // have room for tiles, so that an XCD's workgroups read one k range of the operands together (27 tiles: 8 ranges,
  // 9 tiles: 24), or, from 33 tiles, the number of ranges that fills the CUs.
#ifndef TFB_PP_LONGK
#define TFB_PP_LONGK 1
#endif
#ifndef TFB_PP_FEWTILE
#define TFB_PP_FEWTILE 1
#endif
  if (TFB_PP && TFB_PP_LONGK && N % 256 == 0 && M % 256 == 0 && K % 64 == 0 && K / 64 >= 128) {
    const long t256 = (long)(N / 256) * (M / 256), nkt = K / 64, cus = tfb_resident_slots(1);
    int sp = 0;
    if (t256 >= 64) {
      for (int c = 1; c <= 8 && !sp; ++c) {
        if (nkt / c < 32) continue;
        if (c > 1 && (!ws || (long)c * M * N * 4 > ws_bytes)) continue;
        const long items = t256 * c, rounds = (items + cus - 1) / cus;
        if ((double)items >= 0.9 * (double)(rounds * cus)) sp = c;
      }
    } else if (ws && TFB_PP_FEWTILE) {
      sp = gemm_pp_fewtile_splits(t256, nkt, (long)M * N, ws_bytes);
    }
    if (sp == 1 && !out_f32 && !accumulate) {
      EpiStore e{C, (long)N, out_f32, accumulate, alpha};
      return gemm_pp_launch_lay<2, 0, 0, LAYP, LAYQ>(P, Q, N, M, (long)K * 2, 1, e, stream);
    }
    if (sp > 1) {
      EpiSplit e{ws, (long)N, (long)M * N};
      int st = gemm_pp_launch_lay<2, 0, 0, LAYP, LAYQ>(P, Q, N, M, (long)K * 2, sp, e, stream);
      if (st != TFB_OK) return st;
      return splitk_reduce(ws, C, (long)M * N, sp, out_f32, accumulate, stream, nullptr, nullptr, 1.0f, alpha);
    }
  }
  const long tiles = (long)(N / 128) * (M / 128);
  const int splits = ws ? choose_splits(tiles, K / 64, (long)M * N, ws_bytes) : 1;
  // few output tiles: the ring kernel, its k ranges inside the workgroups, or in workgroups of their own where a quarter of the CUs
  // or less have a tile (256 x 1024 x 4096: 13.7 -> 11.6 us)
  if (const int pick = gemm_ring_pick(N, M, K / 64, LAYP == TFB_K_STRIDED && LAYQ == TFB_K_STRIDED)) {
    GemmArgs a = {};
    a.P = P;
    a.Q = Q;
    a.np = N;
    a.nq = M;
    a.nkt = K / 64;
    if (splits == 1 || 4 * (long)(N / 64) * (M / 64) > tfb_resident_slots(1))
      return gemm_ring_launch<EpiStore, 2, LAYP, LAYQ, 0, 0>(pick, a, 1, 1, EpiStore{C, (long)N, out_f32, accumulate, alpha}, stream, splits);
    const int st = gemm_ring_launch<EpiSplit, 2, LAYP, LAYQ, 0, 0>(pick, a, 1, splits, EpiSplit{ws, (long)N, (long)M * N}, stream);
    return st != TFB_OK ? st : splitk_reduce(ws, C, (long)M * N, splits, out_f32, accumulate, stream, nullptr, nullptr, 1.0f, alpha);
  }
  if (splits == 1) {
    EpiStore e{C, (long)N, out_f32, accumulate, alpha};
    // large outputs: the persistent 256 x 256 kernel (same sums in the same order), in any operand layout (the input
    // gradient of the QKV projection, whose weight is read k-strided: 123.6 -> 117.7 us inside the step)
    int st;
    if (!out_f32 && !accumulate && gemm_pp_try<2, LAYP, LAYQ, 0, 0>(P, Q, N, M, (long)K * 2, false, e, stream, st)) return st;
    return gemm_launch<Cfg>(P, Q, N, M, (long)K * 2, 1, LoadIdentity{}, LoadIdentity{}, e, stream);
  }
  EpiSplit e{ws, (long)N, (long)M * N};
  int st = gemm_launch<Cfg>(P, Q, N, M, (long)K * 2, splits, LoadIdentity{}, LoadIdentity{}, e, stream);
  if (st != TFB_OK) return st;
  return splitk_reduce(ws, C, (long)M * N, splits, out_f32, accumulate, stream, nullptr, nullptr, 1.0f, alpha);
}

// The two gradient GEMMs of y = x w^T as jobs of one ring launch: dx = dy w (w read k-strided), dw (+)= dy^T x (both k-strided).
typedef RingJob<TFB_K_STRIDED, TFB_K_CONTIG, 2, 0, 0, true, EpiStore> JobDx;
typedef RingJob<TFB_K_STRIDED, TFB_K_STRIDED, 2, 0, 0, true, EpiStore> JobDw;
// the k ranges run<>() would sum such a contraction in, or 0 where it takes another kernel than the ring (or cuts the ranges into
// workgroups of their own)
inline int ring_ranges(int N, int M, int K, bool strided, long ws_bytes) {
  if (!gemm_ring_pick(N, M, K / 64, strided)) return 0;
  const int splits = ws_bytes > 0 ? choose_splits((long)(N / 128) * (M / 128), K / 64, (long)M * N, ws_bytes) : 1;
  return splits == 1 || 4 * (long)(N / 64) * (M / 64) > tfb_resident_slots(1) ? splits : 0;
}

// out [q][ld] = bf16(D) with the rotary embedding applied to the first rot_cols columns (heads of 2 HALF: y1 = x1 c + x2 s,
// y2 = x2 c - x1 s on the bf16-rounded products, rounded again - what tfb_rope computes from the stored projection).
template <int HALF>
struct EpiStoreRope {
  static constexpr int kPartner = HALF;
  bf16_t* out;
  long ld;
  const bf16_t* cs;  // [T][HALF]
  const bf16_t* sn;
  int T, rot_cols;
  FastDiv d_T;
  struct pre_t {  // the chunk's cos / sin values, requested before the k-loop
    u32x4 c, s;
  };
  __device__ __forceinline__ long table(int p, int q) const { return (long)(q - fastdiv(q, d_T) * T) * HALF + (p & (HALF - 1)); }
  __device__ __forceinline__ const void* at(int p, int q) const { return cs + table(p, q); }
  __device__ __forceinline__ const void* at2(int p, int q) const { return sn + table(p, q); }
  __device__ __forceinline__ pre_t prefetch(int p, int q) const {
    pre_t r = {};
    if (p < rot_cols) {
      r.c = *(const u32x4*)at(p, q);
      r.s = *(const u32x4*)at2(p, q);
    }
    return r;
  }
  __device__ __forceinline__ void operator()(int p, int q, const float (&v)[8], const float (&vp)[8], const pre_t& tab,
                                             int) const {
    u32x4 x = pack8bf(v);
    if (p < rot_cols) {
      const u32x4 y = pack8bf(vp);
      const bool low = (p & HALF) == 0;
      const u32x4 c = tab.c, s = tab.s;
      u32x4 o;
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float x0 = bflo(x[k]), x1 = bfhi(x[k]), y0 = bflo(y[k]), y1 = bfhi(y[k]);
        const float c0 = bflo(c[k]), c1 = bfhi(c[k]), s0 = bflo(s[k]), s1 = bfhi(s[k]);
        o[k] = low ? pack2bf(x0 * c0 + y0 * s0, x1 * c1 + y1 * s1) : pack2bf(x0 * c0 - y0 * s0, x1 * c1 - y1 * s1);
      }
      x = o;
    }
    *(u32x4*)(out + (long)q * ld + p) = x;
  }
  // the 256 x 256 kernel's protocol: the same from the rounded products, a chunk of a head's first half with its partner
  __device__ __forceinline__ float pre(float x) const { return x; }
  __device__ __forceinline__ void chunk2(int p, int q, u32x4 x, u32x4 y, const u32x4& c, const u32x4& s) const {
    if (p < rot_cols) {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        const float x0 = bflo(x[k]), x1 = bfhi(x[k]), y0 = bflo(y[k]), y1 = bfhi(y[k]);
        const float c0 = bflo(c[k]), c1 = bfhi(c[k]), s0 = bflo(s[k]), s1 = bfhi(s[k]);
        x[k] = pack2bf(x0 * c0 + y0 * s0, x1 * c1 + y1 * s1);
        y[k] = pack2bf(y0 * c0 - x0 * s0, y1 * c1 - x1 * s1);
      }
    }
    bf16_t* o = out + (long)q * ld + p;
    *(u32x4*)o = x;
    *(u32x4*)(o + HALF) = y;
  }
};

template <int HALF>
int qkv_rope(const void* x, const void* w, const void* cos_t, const void* sin_t, void* out, int M, int N, int K, int T, int rot_cols, hipStream_t s) {
  using Cfg = GemmCfg<128, 128, 2, 2, 2, TFB_K_CONTIG, TFB_K_CONTIG>;
  GemmOperand P{(const uint8_t*)w, (long)K * 2}, Q{(const uint8_t*)x, (long)K * 2};
  EpiStoreRope<HALF> e{(bf16_t*)out, (long)N, (const bf16_t*)cos_t, (const bf16_t*)sin_t, T, rot_cols, fastdiv_make(T)};
  int st;
  if (gemm_ring_try<2, TFB_K_CONTIG, TFB_K_CONTIG, 0, 0>(P, Q, N, M, (long)K * 2, e, s, st)) return st;
  if (gemm_pp_try<2, TFB_K_CONTIG, TFB_K_CONTIG, 0, 0>(P, Q, N, M, (long)K * 2, true, e, s, st)) return st;
  return gemm_launch<Cfg>(P, Q, N, M, (long)K * 2, 1, LoadIdentity{}, LoadIdentity{}, e, s);
}

}  // namespace

// tfb_gemm_bf16 with the product multiplied by the device fp32 scalar *alpha (NULL = 1) before its one rounding:
// C (+)= alpha op(A) @ op(B). For gradient GEMMs whose upstream scalar lives on the device.
extern "C" int tfb_gemm_bf16_scaled(const void* A, const void* B, void* C, int M, int N, int K, int trans_a, int trans_b,
                                    int out_f32, int accumulate, void* workspace, long workspace_bytes, const void* alpha,
                                    void* stream) {
  if (!A || !B || !C) return TFB_ERR_ARG;
  if (M <= 0 || N <= 0 || K <= 0 || M % 128 || N % 128 || K % 64) return TFB_ERR_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  // The output's contiguous dimension (n) rides the P side of the core.
  GemmOperand P, Q;
  P.base = (const uint8_t*)B;
  Q.base = (const uint8_t*)A;
  P.ld = trans_b ? (long)K * 2 : (long)N * 2;
  Q.ld = trans_a ? (long)M * 2 : (long)K * 2;
  float* ws = (float*)workspace;
  const float* al = (const float*)alpha;
  if (trans_b && !trans_a) return run<TFB_K_CONTIG, TFB_K_CONTIG>(P, Q, N, M, K, C, out_f32, accumulate, ws, workspace_bytes, al, s);
  if (!trans_b && !trans_a) return run<TFB_K_STRIDED, TFB_K_CONTIG>(P, Q, N, M, K, C, out_f32, accumulate, ws, workspace_bytes, al, s);
  if (!trans_b && trans_a) return run<TFB_K_STRIDED, TFB_K_STRIDED>(P, Q, N, M, K, C, out_f32, accumulate, ws, workspace_bytes, al, s);
  return run<TFB_K_CONTIG, TFB_K_STRIDED>(P, Q, N, M, K, C, out_f32, accumulate, ws, workspace_bytes, al, s);
}

extern "C" int tfb_gemm_bf16(const void* A, const void* B, void* C, int M, int N, int K, int trans_a, int trans_b,
                             int out_f32, int accumulate, void* workspace, long workspace_bytes, void* stream) {
  return tfb_gemm_bf16_scaled(A, B, C, M, N, K, trans_a, trans_b, out_f32, accumulate, workspace, workspace_bytes, nullptr, stream);
}

// TFB_OK where tfb_linear_bwd takes the gradients of M rows through a linear layer w [N][K]: both GEMMs are launches of few tiles, and
// together they have no more than two 128 x 64 tiles for a CU (beyond, two operands' rows displace each other in the L2s: 2048 rows, N
// 3072, K 1024, 640 tiles: two calls 43 us, one 47; 4096 rows, N 2304, K 768, 600 tiles: 50 us either way; 504 tiles: 45 -> 32).
extern "C" int tfb_linear_bwd_applies(int M, int N, int K, long workspace_bytes) {
  if (M <= 0 || N <= 0 || K <= 0 || M % 128 || N % 128 || K % 128) return TFB_ERR_SHAPE;
  if ((long)(K / 128) * (M / 64) + (long)(K / 128) * (N / 64) > 2L * tfb_resident_slots(1)) return TFB_ERR_SHAPE;
  return ring_ranges(K, M, N, false, workspace_bytes) > 0 && ring_ranges(K, N, M, true, workspace_bytes) > 0 ? TFB_OK : TFB_ERR_SHAPE;
}

// The gradients of y [M][N] = x [M][K] @ w [N][K]^T from dy [M][N] in one launch: dx [M][K] = dy @ w, dw [N][K] (+)= dy^T @ x, each
// equal bit for bit to its tfb_gemm_bf16 call with a workspace of workspace_bytes (whose k ranges it sums; none is used here).
// us, two calls -> this one, K 768: 2048 rows, N 2304 31.0 -> 26.5, N 768 16.8 -> 13.9; 1024 rows, N 768 11.0 -> 8.4.
extern "C" int tfb_linear_bwd(const void* dy, const void* x, const void* w, void* dx, void* dw, int M, int N, int K, int dw_f32,
                              int dw_accumulate, long workspace_bytes, void* stream) {
  if (!dy || !x || !w || !dx || !dw) return TFB_ERR_ARG;
  if (tfb_linear_bwd_applies(M, N, K, workspace_bytes) != TFB_OK) return TFB_ERR_SHAPE;
  const GemmOperand W{(const uint8_t*)w, (long)K * 2}, X{(const uint8_t*)x, (long)K * 2}, G{(const uint8_t*)dy, (long)N * 2};
  const JobDx jx(W, G, K, M, (long)N * 2, EpiStore{dx, (long)K, 0, 0}, ring_ranges(K, M, N, false, workspace_bytes));
  const JobDw jw(X, G, K, N, (long)M * 2, EpiStore{dw, (long)K, dw_f32, dw_accumulate}, ring_ranges(K, N, M, true, workspace_bytes));
  return gemm_ring_jobs(jx, jw, (hipStream_t)stream);
}

// C [M][N] = bf16(res + bf16(A [M][K] @ op(B))), B [N][K] (trans_b) or [K][N]: a projection with the residual add that
// follows it made in the store. Equal to tfb_gemm_bf16 followed by a bf16 add, bit for bit. The bf16 form of the
// reference's projection-with-residual forward (round2/source/kernels/nki_attn_nr8.py:1003).
extern "C" int tfb_gemm_bf16_res(const void* A, const void* B, const void* res, void* C, int M, int N, int K, int trans_b,
                                 void* stream) {
  if (!A || !B || !res || !C) return TFB_ERR_ARG;
  if (M <= 0 || N <= 0 || K <= 0 || M % 128 || N % 128 || K % 64) return TFB_ERR_SHAPE;
  GemmOperand P{(const uint8_t*)B, trans_b ? (long)K * 2 : (long)N * 2}, Q{(const uint8_t*)A, (long)K * 2};
  EpiStoreRes e{(bf16_t*)C, (const bf16_t*)res, (long)N};
  int st;
  if (trans_b ? gemm_ring_try<2, TFB_K_CONTIG, TFB_K_CONTIG, 0, 0>(P, Q, N, M, (long)K * 2, e, (hipStream_t)stream, st)
              : gemm_ring_try<2, TFB_K_STRIDED, TFB_K_CONTIG, 0, 0>(P, Q, N, M, (long)K * 2, e, (hipStream_t)stream, st))
    return st;
  if (trans_b && gemm_pp_try<2, TFB_K_CONTIG, TFB_K_CONTIG, 0, 0>(P, Q, N, M, (long)K * 2, true, e, (hipStream_t)stream, st)) return st;
  if (trans_b)
    return gemm_launch<GemmCfg<128, 128, 2, 2, 2, TFB_K_CONTIG, TFB_K_CONTIG>>(P, Q, N, M, (long)K * 2, 1, LoadIdentity{},
                                                                               LoadIdentity{}, e, (hipStream_t)stream);
  return gemm_launch<GemmCfg<128, 128, 2, 2, 2, TFB_K_STRIDED, TFB_K_CONTIG>>(P, Q, N, M, (long)K * 2, 1, LoadIdentity{},
                                                                              LoadIdentity{}, e, (hipStream_t)stream);
}

// qkv [M][N] = rope(x [M][K] @ w [N][K]^T): the fused attention projection with the rotary embedding of the q and k
// thirds (the first rot_cols columns, heads of D = 64 or 128 elements) applied in the GEMM epilogue; row m is token m % T.
// cos_t, sin_t: bf16 [T][D / 2]. The output equals tfb_gemm_bf16 followed by tfb_rope bit for bit. us, two launches -> one, D = 128:
// 512 -> 1536 columns: 1152 rows 9.4 -> 6.8, 4096 18.6 -> 13.8, 12288 36.8 -> 30.9; 1024 -> 3072: 256 8.8 -> 8.2, 1152 17.1 -> 13.5, 6144 55.4 -> 48.5,
// 9600 76.9 -> 72.9, 16384 113 -> 100. Where the projection alone takes tiles that fill its rounds better, which have no rotation, two launches gain
// or lose a little (12288 93.3 -> 95.8; 768 -> 2304: 9600 49.2 -> 50.4, 4096 27.2 -> 27.5).
extern "C" int tfb_qkv_rope_heads_fwd(const void* x, const void* w, const void* cos_t, const void* sin_t, void* out, int M, int N,
                                      int K, int T, int rot_cols, int D, void* stream) {
  if (!x || !w || !cos_t || !sin_t || !out) return TFB_ERR_ARG;
  if ((D != 64 && D != 128) || M <= 0 || N <= 0 || K <= 0 || M % 128 || N % 128 || K % 64 || T <= 0 || rot_cols < 0 || rot_cols > N ||
      rot_cols % D)
    return TFB_ERR_SHAPE;
  return D == 64 ? qkv_rope<32>(x, w, cos_t, sin_t, out, M, N, K, T, rot_cols, (hipStream_t)stream)
                 : qkv_rope<64>(x, w, cos_t, sin_t, out, M, N, K, T, rot_cols, (hipStream_t)stream);
}
extern "C" int tfb_qkv_rope_fwd(const void* x, const void* w, const void* cos_t, const void* sin_t, void* out, int M, int N,
                                int K, int T, int rot_cols, void* stream) {
  return tfb_qkv_rope_heads_fwd(x, w, cos_t, sin_t, out, M, N, K, T, rot_cols, 64, stream);
}
