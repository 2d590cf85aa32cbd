// Symmetric products of a stack of matrices: D = X X^T (or X^T X), bf16 in and out, one 128 x 128 tile per workgroup on and above the
// diagonal, stored a second time transposed above it. Operand layouts, fragments and epilogue protocol are the ring kernel's
// (gemm_ring.hpp), whose 64 x 64 tiles take the small stacks.
//
// What bounds such a tile on one wavefront per SIMD is everything in turn: a CU moves some 85 KB a microsecond into LDS (the loads alone
// of 12 x 768 x 768 over 3072 take 18 us), the MFMAs take 12, the fragment reads, the epilogue. Here eight wavefronts share the tile: two
// groups of four, one of each on every SIMD. Group g multiplies the k-steps 2 g and 2 g + 1 of every k-tile into accumulators of its own
// and issues half of the loads; the groups alternate between a LOAD cluster (four loads of the k-tile three ahead) and an MFMA cluster (8
// MFMAs of 32 x 32, the next k-tile's fragments read between them), group 1 one cluster behind group 0. The two partial sums meet in LDS
// at the end (sum of group 0 + sum of group 1, the order gemm_ring_tile keeps for these epilogues too; against 64 bits no worse than one
// chain, half of its error where the sums have a mean), and a tile above the diagonal is transposed by transposing LDS reads
// (MirrorBlock). us, four wavefronts -> this: 12 x 768 x 768 over 3072 34.8 -> 30, over 768 15.0 -> 13; five iterations of 24 x 3072 x 768
// 1069 -> 1031 (the chip's power limit takes the rest: the same launches on zeros run in 0.8 of the time).
//
// Slots between barriers, k-tile t: group 0 LOAD 2 t, MFMA 2 t + 1; group 1 LOAD 2 t + 1, MFMA 2 t + 2. Stage (t + 1) % 4 is read in slots
// 2 t + 1 and 2 t + 2, its reads waited for in front of the barriers that end slots 2 t + 2 and 2 t + 3, and requested again (k-tile t + 5)
// in slots 2 t + 4 and 2 t + 5. K-tile t + 1 has to be there at the barrier that ends slot 2 t: group 0 waits for its loads at the end of LOAD t,
// group 1 at the end of MFMA t - 1.
#pragma once
#include "gemm_ring.hpp"

struct SymArgs {
  GemmOperand X;
  long g_stride;   // the operand of group g starts g_stride bytes * g further
  int nkt;         // k-tiles of 64: an even number
  int nt;          // tiles of a side
  int ntiles, groups, per;   // nt (nt + 1) / 2 tiles a group; XCD x (= workgroup & 7) takes `per` consecutive tiles of the stack
  FastDiv d_ntiles;
};

// A wavefront's fragments of two k-steps of one operand's 64 rows: request() asks for them, landed() ties them to the wait before it.
template <int LAY>
struct SymFrags;
template <>
struct SymFrags<TFB_K_CONTIG> {
  i32x4 v[2][2];   // [MFMA tile][k-step]
  static __device__ __forceinline__ void addr(uint32_t (&a)[2], int row0, int lane, int g) {
    const int row = row0 + (lane & 31), lh = lane >> 5;
#pragma unroll
    for (int s = 0; s < 2; ++s) a[s] = row * 128 + ((((2 * (2 * g + s) + lh) ^ tfb_kc_swz(row)) & 7) << 4);
  }
  // reads 2 m and 2 m + 1 of the operand's, m = 0 .. 3 (a 128-bit read counts as two)
  template <int m>
  __device__ __forceinline__ void request(const uint32_t (&a)[2], uint32_t base) {
    v[m & 1][m >> 1] = ring_read128<4096 * (m & 1)>(base + a[m >> 1]);
  }
  __device__ __forceinline__ void landed() { asm volatile("" : "+v"(v[0][0]), "+v"(v[0][1]), "+v"(v[1][0]), "+v"(v[1][1])); }
  __device__ __forceinline__ bf16x8 get(int i, int s) const { return __builtin_bit_cast(bf16x8, v[i][s]); }
};
template <>
struct SymFrags<TFB_K_STRIDED> {
  u32x2 v[2][2][2];   // [MFMA tile][k-step][k 0-3 / 4-7]
  static __device__ __forceinline__ void addr(uint32_t (&a)[2], int row0, int lane, int g) {
    const int g4 = lane >> 4, j = lane & 15, k = 8 * (g4 >> 1) + (j >> 2);
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      const int p = row0 + 32 * i + 16 * (g4 & 1) + 4 * (j & 3);
      a[i] = (32 * g + k) * 256 + ((((p >> 3) ^ tfb_ks_swz<128, 2>(k)) << 4) | ((p & 4) << 1));
    }
  }
  template <int m>
  __device__ __forceinline__ void request(const uint32_t (&a)[2], uint32_t base) {
    constexpr int i = m & 1, s = m >> 1;
    v[i][s][0] = ring_read_tr64<4096 * s, 2>(base + a[i]);
    v[i][s][1] = ring_read_tr64<4096 * s + 1024, 2>(base + a[i]);
  }
  __device__ __forceinline__ void landed() {
#pragma unroll
    for (int i = 0; i < 2; ++i) asm volatile("" : "+v"(v[i][0][0]), "+v"(v[i][0][1]), "+v"(v[i][1][0]), "+v"(v[i][1][1]));
  }
  __device__ __forceinline__ bf16x8 get(int i, int s) const {
    const u32x4 w = {v[i][s][0].x, v[i][s][0].y, v[i][s][1].x, v[i][s][1].y};
    return __builtin_bit_cast(bf16x8, w);
  }
};

template <int LAY, class Epi>
__global__ __launch_bounds__(512, 2) void gemm_sym_kernel(SymArgs a, Epi epi_in) {
  constexpr int NS = 4, STAGE = 32768, SLD = 68, LDS = NS * STAGE;
  typedef MirrorBlock<64> Mirror;
  constexpr int EPI = 32 * SLD * 4 + Mirror::OUT_BYTES;   // of a wavefront: 32 x 64 in fp32 (then bf16, for the mirror), the transposed block
  static_assert(8 * EPI <= LDS && Mirror::BYTES <= 32 * SLD * 4, "epilogue slices");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[LDS];
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int g = wave >> 2, wp = wave & 1, wq = (wave >> 1) & 1;   // wavefronts w and w + 4 share a SIMD
  const int lr = lane & 31, lh = lane >> 5;
  const int lid = (blockIdx.x & 7) * a.per + (blockIdx.x >> 3);
  const int group = fastdiv(lid, a.d_ntiles);
  if (group >= a.groups) return;   // (the whole workgroup: the XCDs' runs are of equal length)
  int tile_p = lid - group * a.ntiles, tile_q = 0;
  for (; tile_p >= a.nt - tile_q; ++tile_q) tile_p -= a.nt - tile_q;   // row tile_q has nt - tile_q tiles
  tile_p += tile_q;
  const int p0 = tile_p * 128, q0 = tile_q * 128;
  const int nkt = a.nkt;
  GemmOperand X = a.X;
  X.base += group * a.g_stride;

  TileDma<128, 8, LAY, 2> dp, dq;
  dp.init(X, p0, 0, wave, lane);
  dq.init(X, q0, 0, wave, lane);
  auto issue = [&](int t) __attribute__((always_inline)) {   // four loads a wavefront
    uint8_t* d = lds + (t & (NS - 1)) * STAGE;
    dp.issue(d, t, wave);
    dq.issue(d + 16384, t, wave);
  };
  for (int t = 0; t < NS - 1; ++t)
    if (t < nkt) issue(t);

  const Epi epi = epi_prepare(epi_for_group(epi_in, group));
  uint32_t ap[2], aq[2];
  SymFrags<LAY>::addr(ap, wp * 64, lane, g);
  SymFrags<LAY>::addr(aq, wq * 64, lane, g);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(tfb_lds_void_t*)lds;
  SymFrags<LAY> fp[2], fq[2];
  f32x16 acc[2][2];
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int j = 0; j < 2; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // the epilogue's chunk k of this wavefront, which finishes the 32 rows q of j = g: row and first column in its slice
  constexpr bool kPrefetch = has_prefetch<Epi>::value;
  auto chunk_row = [&](int k) { return 2 * ((lane >> 3) / 2 + 4 * k) + ((lane >> 2) & 1); };
  auto chunk_col = [&](int k) { return (4 * ((lane >> 3) & 1) + (lane & 3)) * 8; };
  const int pw = p0 + wp * 64, qw = q0 + wq * 64 + 32 * g;
  [[maybe_unused]] typename prefetch_type<Epi>::type pre[4];

  if (nkt > 2) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");   // k-tiles 0 and 1 (nkt >= 2)
  else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  TFB_SBAR();
  typedef std::integral_constant<int, 0> N0;
  typedef std::integral_constant<int, 1> N1;
  typedef std::integral_constant<int, 2> N2;
  typedef std::integral_constant<int, 3> N3;
  fp[0].template request<0>(ap, lds0);
  fp[0].template request<1>(ap, lds0);
  fp[0].template request<2>(ap, lds0);
  fp[0].template request<3>(ap, lds0);
  fq[0].template request<0>(aq, lds0 + 16384);
  fq[0].template request<1>(aq, lds0 + 16384);
  fq[0].template request<2>(aq, lds0 + 16384);
  fq[0].template request<3>(aq, lds0 + 16384);
  if constexpr (kPrefetch) {
#pragma unroll
    for (int k = 0; k < 4; ++k) pre[k] = epi.prefetch(pw + chunk_col(k), qw + chunk_row(k));
  }
  if (g == 1) TFB_SBAR();   // group 1 runs one cluster behind from here on

  // k-tile t, its fragments in set `set`; LEFT = k-tiles behind it, counted up to 3
  auto step = [&](int t, auto SET, auto LEFT) __attribute__((always_inline)) {
    constexpr int set = decltype(SET)::value, left = decltype(LEFT)::value;
    // LOAD
    if constexpr (left == 3) issue(t + 3);
    if constexpr (left > 0) {
      if (g == 0) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (left - 1)) : "memory");
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    fp[set].landed();
    fq[set].landed();
    TFB_SBAR();
    // MFMA: eight of them, two reads of the next k-tile's fragments behind each
    const uint32_t b = lds0 + ((t + 1) & (NS - 1)) * STAGE;
    __builtin_amdgcn_s_setprio(1);
    auto one = [&](auto M) __attribute__((always_inline)) {
      constexpr int m = decltype(M)::value, s = m >> 2, i = (m >> 1) & 1, j = m & 1;
      acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(fp[set].get(i, s), fq[set].get(j, s), acc[i][j], 0, 0, 0);
      if constexpr (left > 0) {
        if constexpr (m & 1) fq[set ^ 1].template request<(m >> 1)>(aq, b + 16384);
        else fp[set ^ 1].template request<(m >> 1)>(ap, b);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    one(N0{});
    one(N1{});
    one(N2{});
    one(N3{});
    one(std::integral_constant<int, 4>{});
    one(std::integral_constant<int, 5>{});
    one(std::integral_constant<int, 6>{});
    one(std::integral_constant<int, 7>{});
    __builtin_amdgcn_s_setprio(0);
    asm volatile("" : "+v"(acc[0][0]), "+v"(acc[0][1]), "+v"(acc[1][0]), "+v"(acc[1][1]));
    if constexpr (left > 1) {
      if (g == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(4 * (left - 2)) : "memory");
    }
    TFB_SBAR();
  };
  int t = 0;
  if (nkt > 4) {
    do {
      step(t, N0{}, N3{});
      step(t + 1, N1{}, N3{});
      t += 2;
    } while (nkt - t > 4);
  }
  if (nkt - t == 4) {
    step(t, N0{}, N3{});
    step(t + 1, N1{}, N2{});
    step(t + 2, N0{}, N1{});
    step(t + 3, N1{}, N0{});
  } else {
    step(t, N0{}, N1{});
    step(t + 1, N1{}, N0{});
  }
  if (g == 0) TFB_SBAR();   // group 0 waits for group 1's last cluster: every stage has been read

  // each wavefront hands the partner on its SIMD the half of its sums that the partner finishes (j = the partner's group)
  f32x16 sum[2];
  {
    f32x4* x = (f32x4*)lds + wave * 512 + lane;
    const f32x4* y = (const f32x4*)lds + (wave ^ 4) * 512 + lane;
    auto hand = [&](auto J) __attribute__((always_inline)) {
      constexpr int j = decltype(J)::value;
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        sum[i] = acc[i][1 - j];
#pragma unroll
        for (int jj = 0; jj < 4; ++jj)
          x[(i * 4 + jj) * 64] = f32x4{acc[i][j][4 * jj], acc[i][j][4 * jj + 1], acc[i][j][4 * jj + 2], acc[i][j][4 * jj + 3]};
      }
    };
    if (g) hand(std::integral_constant<int, 0>{});
    else hand(std::integral_constant<int, 1>{});
    __syncthreads();
#pragma unroll
    for (int i = 0; i < 2; ++i)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const f32x4 o = y[(i * 4 + jj) * 64];
#pragma unroll
        for (int e = 0; e < 4; ++e) sum[i][4 * jj + e] += o[e];
      }
    __syncthreads();
  }
  // 32 rows q x 64 p through the wavefront's own slice, then 8-element chunks, a row's on consecutive lanes; above the diagonal once more
  // as 64-byte pieces of the rows p
  uint8_t* area = lds + wave * EPI;
  float* stg = (float*)area;
#pragma unroll
  for (int i = 0; i < 2; ++i)
#pragma unroll
    for (int jj = 0; jj < 4; ++jj) {
      const f32x4 v = {sum[i][jj * 4 + 0], sum[i][jj * 4 + 1], sum[i][jj * 4 + 2], sum[i][jj * 4 + 3]};
      *(f32x4*)(stg + lr * SLD + i * 32 + jj * 8 + lh * 4) = v;
    }
  __builtin_amdgcn_wave_barrier();
  u32x4 w[4];
#pragma unroll
  for (int k = 0; k < 4; ++k) {
    const int row = chunk_row(k), pc = chunk_col(k);
    const f32x4 lo = *(const f32x4*)(stg + row * SLD + pc), hi = *(const f32x4*)(stg + row * SLD + pc + 4);
    const float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
    if constexpr (kPrefetch) w[k] = epi.value(v, pre[k]);
    else w[k] = epi.value(v);
    *(u32x4*)(epi.out + (long)(qw + row) * epi.ld + pw + pc) = w[k];
  }
  if (tile_p != tile_q) {
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < 4; ++k) Mirror::put(area, chunk_row(k), chunk_col(k), w[k]);
    Mirror::store(area, area + 32 * SLD * 4, epi.out + (long)pw * epi.ld + qw, epi.ld, lane);
  }
}

// A stack of `groups` symmetric N x N products of one operand with itself (N and the contraction multiples of 128): 64 x 64
// tiles of the ring kernel while no CU has more than two, else 128 x 128 (half the bytes per output, one workgroup per CU). An XCD's
// workgroups take a run of consecutive tiles, so that a matrix's operand is read into one or two L2s only.
template <class Epi, int LAY>
static int gemm_symmetric(GemmOperand X, long g_stride, int N, int nkt, int groups, Epi e, hipStream_t s) {
  if (N <= 0 || N % 128 || groups <= 0 || nkt < 2 || nkt % 2) return TFB_ERR_SHAPE;
  const long n64 = N / 64, cus = tfb_resident_slots(1);
  if (n64 * (n64 + 1) / 2 * groups <= 2 * cus) return gemm_ring_symmetric<Epi, 2, LAY>(X, g_stride, N, nkt, groups, e, s);
  if (X.ld <= 0 || X.ld > (1L << 28)) return TFB_ERR_SHAPE;
  if (((uintptr_t)X.base | (uintptr_t)X.ld) & 15) return TFB_ERR_ARG;
  SymArgs a = {X, g_stride, nkt, N / 128, 0, groups, 0, {}};
  a.ntiles = a.nt * (a.nt + 1) / 2;
  if ((long)a.ntiles * groups > 0x7ffffff0L / 8) return TFB_ERR_SHAPE;
  a.per = (a.ntiles * groups + 7) / 8;
  a.d_ntiles = fastdiv_make(a.ntiles);
  hipLaunchKernelGGL((gemm_sym_kernel<LAY, Epi>), dim3(8 * a.per), dim3(512), 0, s, a, e);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}
