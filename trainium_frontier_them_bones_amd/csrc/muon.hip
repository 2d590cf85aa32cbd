// Muon's Newton-Schulz ("Polar Express") orthogonalisation of a stack of gradient matrices, five iterations, bf16 with
// fp32 accumulation. Replaces _nsk_kernel (round2/source/kernels/nki_nsk.py:370; arithmetic: emulate_nsk 452, _ns_tall 426)
// and the loop of muon_math_body it restates (reference_ns, nki_nsk.py:471).
//
// Per matrix, held tall X [M][N] (M >= N; a wide input [N][M] is transposed on the way in and out):
//   X0 = bf16(bf16(g) * (1 / d))
//   G  = bf16(X^T X)                          [N][N]   contraction over the M rows
//   B  = bf16(fp32(G G * c) + fp32(b * G))    [N][N]   one rounding
//   X' = bf16(fp32(X B) + fp32(a * X))        [M][N]   one rounding
// with the five (a, b, c) of the caller, then v[m] = sum_n X5[m][n]^2 in fp32 from the bf16 X5.
//
// The whole stack runs in three grouped GEMM launches per iteration (not three per matrix): the matrices are stacked
// along the rows, G's contraction is over a matrix's own rows, and X B picks the [N][N] operand by the row tile's matrix
// (q_group). G and G G are symmetric bit for bit (the same products summed in the same order on either side of the
// diagonal): their tiles on and above the diagonal are computed, those above it stored a second time transposed, and with
// B^T = B both products run in the k-contiguous "x @ w^T" form with the [N][N] matrix as the weight.
#include "gemm_sym.hpp"

extern "C" long tfb_ns5_workspace_bytes(int K, int M, int N);

namespace {

__device__ __forceinline__ u32x4 axpby8(const float (&v)[8], const u32x4& zv, float alpha, float beta) {
  float zf[8], r[8];
  unpack8bf(zv, zf);
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float t1 = v[k] * alpha, t2 = beta * zf[k];
    r[k] = t1 + t2;
  }
  return pack8bf(r);
}

// out = bf16(fp32(alpha * D) + fp32(beta * z)), z and out [rows][ld] bf16; the z chunk is requested before the k-loop. Rows from `split` on
// go to out2 (at the same offsets)
struct EpiAxpby {
  bf16_t* out;
  bf16_t* out2;
  int split;
  const bf16_t* z;
  long ld;
  float alpha, beta;
  using pre_t = u32x4;
  __device__ __forceinline__ pre_t prefetch(int p, int q) const { return *(const u32x4*)(z + (long)q * ld + p); }
  __device__ __forceinline__ void operator()(int p, int q, const float (&v)[8], const pre_t& zv, int) const {
    *(u32x4*)((q < split ? out : out2) + (long)q * ld + p) = axpby8(v, zv, alpha, beta);
  }
};

// A symmetric product of the stack, bf16 [K][N][N]: out = bf16(D), or bf16(fp32(alpha D) + fp32(beta z))
struct EpiSym {
  static constexpr bool kSymmetric = true;
  bf16_t* out;
  long ld, slab;
  __device__ __forceinline__ EpiSym for_group(int g) const { return EpiSym{out + g * slab, ld, slab}; }
  __device__ __forceinline__ u32x4 value(const float (&v)[8]) const { return pack8bf(v); }
};
struct EpiSymAxpby {
  static constexpr bool kSymmetric = true;
  bf16_t* out;
  const bf16_t* z;
  long ld, slab;
  float alpha, beta;
  using pre_t = u32x4;
  __device__ __forceinline__ EpiSymAxpby for_group(int g) const { return EpiSymAxpby{out + g * slab, z + g * slab, ld, slab, alpha, beta}; }
  __device__ __forceinline__ pre_t prefetch(int p, int q) const { return *(const u32x4*)(z + (long)q * ld + p); }
  __device__ __forceinline__ u32x4 value(const float (&v)[8], const pre_t& zv) const {
    return axpby8(v, zv, alpha, beta);
  }
};

// The reciprocals of a stack's denominators: what the caller computed, or 1 / fp32(d) of its denominators
#define NS_INV 0
#define NS_D_F32 1
#define NS_D_BF16 2
#define NS_D_F16 3
__device__ __forceinline__ float ns_inverse(const void* d, int type, int k) {
  if (type == NS_INV) return ((const float*)d)[k];
  if (type == NS_D_F32) return 1.0f / ((const float*)d)[k];
  if (type == NS_D_BF16) return 1.0f / __uint_as_float((uint32_t)((const bf16_t*)d)[k] << 16);
  return 1.0f / (float)((const _Float16*)d)[k];
}

// X0 [K][M][N] bf16 = bf16(bf16(g) * inv_d[k]); g fp32 [K][M][N], or with WIDE [K][N][M] (32 x 32 tiles through LDS). Also the table of the
// matrix that a row tile of 128 belongs to: xq[k M / 128 ..] = first + k.
template <bool WIDE>
__global__ __launch_bounds__(256) void ns_load_kernel(const float* __restrict__ g, const void* __restrict__ d, int type,
                                                     bf16_t* __restrict__ x, int* __restrict__ xq, int first, int M, int N) {
  const int k = blockIdx.z;
  const float r = ns_inverse(d, type, k);
  const long mat = (long)k * M * N;
  if (blockIdx.x == 0 && blockIdx.y == 0)
    for (int i = threadIdx.x; i < M / 128; i += 256) xq[k * (M / 128) + i] = first + k;
  if (!WIDE) {
    const long n = (long)M * N;
    for (long i = ((long)blockIdx.x * 256 + threadIdx.x) * 4; i < n; i += (long)gridDim.x * 256 * 4) {
      const f32x4 v = *(const f32x4*)(g + mat + i);
      u32x2 o = {pack2bf(round_bf(v[0]) * r, round_bf(v[1]) * r), pack2bf(round_bf(v[2]) * r, round_bf(v[3]) * r)};
      *(u32x2*)(x + mat + i) = o;
    }
  } else {
    __shared__ float t[32][33];
    const int m0 = blockIdx.x * 32, n0 = blockIdx.y * 32;  // tile of the tall X: rows m0.., columns n0..
    const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
#pragma unroll
    for (int j = 0; j < 32; j += 8) t[ty + j][tx] = g[mat + (long)(n0 + ty + j) * M + m0 + tx];  // g[n][m]
    __syncthreads();
#pragma unroll
    for (int j = 0; j < 32; j += 8) x[mat + (long)(m0 + ty + j) * N + n0 + tx] = f2bf(round_bf(t[tx][ty + j]) * r);
  }
}

// v[k][m] = sum_n X[k][m][n]^2 (fp32, from the bf16 values): one wavefront per row. Rows from `split` on are x2's and go to v2 (at the
// same offsets).
__global__ __launch_bounds__(256) void ns_rowsq_kernel(const bf16_t* __restrict__ x, const bf16_t* __restrict__ x2, float* __restrict__ v,
                                                      float* __restrict__ v2, long split, long rows, int N) {
  const int lane = threadIdx.x & 63;
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  if (row >= split) {
    x = x2;
    v = v2;
  }
  float s = 0.f;
  for (int c = lane * 8; c < N; c += 512) {
    float f[8];
    unpack8bf(*(const u32x4*)(x + row * N + c), f);
#pragma unroll
    for (int k = 0; k < 8; ++k) s += f[k] * f[k];
  }
  s = wave_sum(s);
  if (lane == 0) v[row] = s;
}

// y [K][N][M] = X [K][M][N]^T (bf16), 32 x 32 tiles through LDS
__global__ __launch_bounds__(256) void ns_transpose_out_kernel(const bf16_t* __restrict__ x, bf16_t* __restrict__ y, int M, int N) {
  __shared__ bf16_t t[32][34];
  const long mat = (long)blockIdx.z * M * N;
  const int m0 = blockIdx.x * 32, n0 = blockIdx.y * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;
#pragma unroll
  for (int j = 0; j < 32; j += 8) t[ty + j][tx] = x[mat + (long)(m0 + ty + j) * N + n0 + tx];
  __syncthreads();
#pragma unroll
  for (int j = 0; j < 32; j += 8) y[mat + (long)(n0 + ty + j) * M + m0 + tx] = t[tx][ty + j];
}

// A grouped launch of `nkt` k-tiles a matrix: the ring kernel for a small stack, else the 128 x 128 core.
template <class Cfg, class Epi>
int launch(const GemmArgs& a, int groups_y, int nkt, Epi e, hipStream_t s) {
  if (const int pick = gemm_ring_pick(a.np, a.nq, nkt, Cfg::LAYP == TFB_K_STRIDED, groups_y))
    return gemm_ring_launch<Epi, 2, Cfg::LAYP, Cfg::LAYQ, 0, 0>(pick, a, groups_y, 1, e, s);
  return gemm_launch_args<Cfg>(a, groups_y, 1, LoadIdentity{}, LoadIdentity{}, e, s);
}

inline long align256(long b) { return (b + 255) & ~255L; }

}  // namespace

namespace {

struct NsStack {   // K matrices of one layout; d: their reciprocals or denominators (NS_*)
  const void *g, *d;
  void *y, *v;
  int K, wide;
};

// Both stacks, the matrices of A in front of B's: one launch of every kind for all of them (a stack of few matrices leaves most CUs idle: 1 + 1
// matrices of 3072 x 768, their reciprocals included, in two calls 326 us, in one 193), a stack's own only where its layout differs.
int ns_run(const NsStack& A, const NsStack& B, int d_type, const float* coeffs, int M, int N, void* workspace, long workspace_bytes, hipStream_t s) {
  const int K = A.K + B.K;
  if (!A.g || !A.d || !A.y || !A.v || (B.K && (!B.g || !B.d || !B.y || !B.v)) || !coeffs || !workspace) return TFB_ERR_ARG;
  if (A.K <= 0 || B.K < 0 || M <= 0 || N <= 0 || M % 128 || N % 128 || M < N || (long)A.K + B.K > 65535 || (long)K * M > 0x7fffffffL / 2) return TFB_ERR_SHAPE;
  if (workspace_bytes < tfb_ns5_workspace_bytes(K, M, N)) return TFB_ERR_WORKSPACE;
  uint8_t* w = (uint8_t*)workspace;
  const long xb = align256((long)K * M * N * 2), gb = align256((long)K * N * N * 2), mat = (long)M * N;
  bf16_t* X[2] = {(bf16_t*)w, (bf16_t*)(w + xb)};
  bf16_t* G = (bf16_t*)(w + 2 * xb);
  bf16_t* Bm = (bf16_t*)(w + 2 * xb + gb);
  int* xq = (int*)(w + 2 * xb + 2 * gb);

  auto load = [&](const NsStack& S, int first) {
    if (S.K == 0) return TFB_OK;
    if (S.wide)
      hipLaunchKernelGGL(ns_load_kernel<true>, dim3(M / 32, N / 32, S.K), dim3(256), 0, s, (const float*)S.g, S.d, d_type, X[0] + first * mat,
                         xq + first * (M / 128), first, M, N);
    else
      hipLaunchKernelGGL(ns_load_kernel<false>, dim3(256, 1, S.K), dim3(256), 0, s, (const float*)S.g, S.d, d_type, X[0] + first * mat,
                         xq + first * (M / 128), first, M, N);
    TFB_LAUNCH_CHECK();
    return TFB_OK;
  };
  int st = load(A, 0);
  if (st == TFB_OK) st = load(B, A.K);
  if (st != TFB_OK) return st;

  using CfgN = GemmCfg<128, 128, 2, 2, 2, TFB_K_CONTIG, TFB_K_CONTIG>;
  bf16_t *x5a = nullptr, *x5b = nullptr;   // the last iterate's rows of either stack, from row 0 of all of them
  for (int it = 0; it < 5; ++it) {
    const float a = coeffs[3 * it], b = coeffs[3 * it + 1], c = coeffs[3 * it + 2];
    bf16_t *xin = X[it & 1], *xout = X[(it & 1) ^ 1];
    // a tall stack's last iteration writes y itself
    x5a = it == 4 && !A.wide ? (bf16_t*)A.y : xout;
    x5b = it == 4 && B.K && !B.wide ? (bf16_t*)B.y - A.K * mat : xout;
    // G[k] = X[k]^T X[k]: both operands k-strided (rows of X[k])
    st = gemm_symmetric<EpiSym, TFB_K_STRIDED>(GemmOperand{(const uint8_t*)xin, (long)N * 2}, mat * 2, N, M / 64, K, EpiSym{G, (long)N, (long)N * N}, s);
    if (st != TFB_OK) return st;
    // B = c G G + b G: G[k] against itself (G G^T = G G)
    st = gemm_symmetric<EpiSymAxpby, TFB_K_CONTIG>(GemmOperand{(const uint8_t*)G, (long)N * 2}, (long)N * N * 2, N, N / 64, K,
                                                   EpiSymAxpby{Bm, G, (long)N, (long)N * N, c, b}, s);
    if (st != TFB_OK) return st;
    // X' = X B + a X on the stacked X: rows of X[k] against B[k] as the weight (X B^T = X B)
    GemmArgs gx;
    gx.P = GemmOperand{(const uint8_t*)Bm, (long)N * 2};
    gx.Q = GemmOperand{(const uint8_t*)xin, (long)N * 2};
    gx.np = N;
    gx.nq = K * M;
    gx.nkt = N * 2 / 128;
    gx.ntp = N / 128;
    gx.q_group = xq;
    gx.p_group_stride = (long)N * N * 2;
    gx.k_seg = nullptr;
    st = launch<CfgN>(gx, 1, gx.nkt, EpiAxpby{x5a, x5b, A.K * M, xin, (long)N, 1.0f, a}, s);
    if (st != TFB_OK) return st;
  }
  const long rows = (long)K * M, split = (long)A.K * M;
  hipLaunchKernelGGL(ns_rowsq_kernel, dim3((unsigned)((rows + 3) / 4)), dim3(256), 0, s, x5a, x5b, (float*)A.v, (float*)B.v - split, split, rows, N);
  TFB_LAUNCH_CHECK();
  auto transpose = [&](const NsStack& S, const bf16_t* x5) {
    if (S.K == 0 || !S.wide) return TFB_OK;
    hipLaunchKernelGGL(ns_transpose_out_kernel, dim3(M / 32, N / 32, S.K), dim3(256), 0, s, x5, (bf16_t*)S.y, M, N);
    TFB_LAUNCH_CHECK();
    return TFB_OK;
  };
  st = transpose(A, x5a);
  return st != TFB_OK ? st : transpose(B, x5b + A.K * mat);
}

}  // namespace

// Bytes of device workspace tfb_ns5 needs for a stack of K matrices (tfb_ns5_stacks: of both stacks' together) with long side M and short side N.
extern "C" long tfb_ns5_workspace_bytes(int K, int M, int N) {
  if (K <= 0 || M <= 0 || N <= 0) return 0;
  const long xb = align256((long)K * M * N * 2), gb = align256((long)K * N * N * 2);
  return 2 * xb + 2 * gb + align256((long)K * (M / 128) * 4);
}

// g: fp32 [K][M][N] (wide = 0) or [K][N][M] (wide = 1: each matrix is handled as its transpose), M >= N; inv_d: fp32 [K]
// device (1 / d of each matrix, d as the caller's optimizer computes it); coeffs: 15 HOST floats, (a, b, c) of the five
// iterations; y: bf16, the layout of g; v: fp32 [K][M]. M, N multiples of 128. The call enqueues 2 + 15 (+1) launches
// on `stream` and returns; the workspace must stay untouched until they have run.
extern "C" int tfb_ns5(const void* g, const void* inv_d, const float* coeffs, void* y, void* v, int K, int M, int N, int wide,
                       void* workspace, long workspace_bytes, void* stream) {
  return ns_run(NsStack{g, inv_d, y, v, K, wide}, NsStack{}, NS_INV, coeffs, M, N, workspace, workspace_bytes, (hipStream_t)stream);
}

// tfb_ns5 of two stacks of the same tall shape, each in its own layout, from the denominators themselves (d_type: 1 fp32, 2 bf16, 3 fp16; the
// reciprocal is taken in fp32): every matrix comes out as tfb_ns5 leaves it, bit for bit. Kb 0: one stack, B's pointers may be NULL.
extern "C" int tfb_ns5_stacks(const void* ga, const void* da, void* ya, void* va, int Ka, int wide_a, const void* gb, const void* db, void* yb,
                              void* vb, int Kb, int wide_b, int d_type, const float* coeffs, int M, int N, void* workspace,
                              long workspace_bytes, void* stream) {
  if (d_type != NS_D_F32 && d_type != NS_D_BF16 && d_type != NS_D_F16) return TFB_ERR_ARG;
  return ns_run(NsStack{ga, da, ya, va, Ka, wide_a}, NsStack{gb, db, yb, vb, Kb, wide_b}, d_type, coeffs, M, N, workspace, workspace_bytes, (hipStream_t)stream);
}
