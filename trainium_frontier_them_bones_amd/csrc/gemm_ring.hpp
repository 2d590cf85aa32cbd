// Small-output MFMA GEMM for gfx950: D[p][q] = sum_k P[p][k] * Q[q][k], the arithmetic, operand layouts and epilogues of the
// 128 x 128 core (gemm_core.hpp) for launches that do not fill the chip with large tiles.
//
// What bounds such a launch is latency: with fewer workgroups than CUs nothing hides a k-tile's trip from L2 or HBM into LDS,
// and the core's two-stage loop pays that trip (about a microsecond) once per k-tile. Here the operand tiles go through a RING of
// NS stages with NS - 1 k-tiles in flight, waited for one by one (s_waitcnt vmcnt(n)), and the tile is as small as it takes to
// give every CU work (64 x 64, 128 x 64 or 128 x 128). The fragments of a k-tile are read in one go while the MFMAs of the k-tile
// before run (two register sets), so a step costs one barrier and no exposed LDS latency.
//
// A contraction that the other kernels cut into k-splits (fp32 partials through memory, a reduction launch) is summed here in the
// same ranges inside the workgroup - partial sums into one set of accumulators, folded into a second at a range's end - so that the
// result is theirs bit for bit and does not depend on which kernel a batch size selects.
//
// Reads from LDS are inline assembly with explicit waits: left to the compiler, each would wait for every load in flight into LDS.
#pragma once
#include "gemm_pp.hpp"

#define TFB_MAX_RING 8

// Epilogues of contractions that may be cut into k ranges declare  static constexpr bool kRanges
template <class T, class = void>
struct has_ranges : std::false_type {};
template <class T>
struct has_ranges<T, std::void_t<decltype(T::kRanges)>> : std::true_type {};

// Epilogues of products that are symmetric bit for bit (D[p][q] = D[q][p]: the same operand on both sides, the contraction in the same
// order) declare  static constexpr bool kSymmetric : the launch is one workgroup per tile on and above the diagonal, and a tile above it
// is stored a second time, transposed through LDS. They give  u32x4 value(v [, pre_t])  (eight rounded outputs),  out  and  ld.
template <class T, class = void>
struct is_symmetric : std::false_type {};
template <class T>
struct is_symmetric<T, std::void_t<decltype(T::kSymmetric)>> : std::true_type {};

// A wavefront's 32 (q) x PC (p) block of finished outputs, transposed: out[p][q]. put() takes its 8-element chunks of rows q, store()
// fetches them as columns with ds_read_b64_tr_b16 (a lane: 8 consecutive q of one p) and writes 64-byte pieces of the rows p. Both
// areas are the wavefront's own (LDS operations of one wavefront execute in order); the paddings spread rows over the banks.
// (Element by element, 32 two-byte writes a lane, this was 4 of 31 us of a 12 x 768 x 768 product over 3072.)
template <int PC>
struct MirrorBlock {
  static constexpr int QP = PC * 2 + 16, PP = 80;              // bytes of a row q, of a row p
  static constexpr int BYTES = 32 * QP, OUT_BYTES = PC * PP;
  static __device__ __forceinline__ void put(uint8_t* t, int row, int pc, const u32x4& w) { *(u32x4*)(t + row * QP + pc * 2) = w; }
  static __device__ __forceinline__ void store(const uint8_t* t, uint8_t* o, bf16_t* out, long ld, int lane) {
    const int g4 = lane >> 4, j = lane & 15;
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int r = 0; r < PC / 16; ++r) {   // lane group g4: rows p 16 r .. + 15, q 8 g4 .. + 7
      const uint8_t* a = t + (8 * g4 + (j >> 2)) * QP + 32 * r + 8 * (j & 3);
      const tfb_s16x4 lo = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tfb_lds_s16x4_t*)a);
      const tfb_s16x4 hi = __builtin_amdgcn_ds_read_tr16_b64_v4i16((tfb_lds_s16x4_t*)(a + 4 * QP));
      typedef short s16x8 __attribute__((ext_vector_type(8)));
      *(s16x8*)(o + (16 * r + j) * PP + 16 * g4) = s16x8{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
    }
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int k = 0; k < PC / 16; ++k) {
      const int row = (lane >> 2) + 16 * k, qc = (lane & 3) * 16;
      *(u32x4*)((uint8_t*)(out + (long)row * ld) + qc) = *(const u32x4*)(o + row * PP + qc);
    }
    __builtin_amdgcn_wave_barrier();
  }
};

template <int BP_, int BQ_, int WP_, int WQ_, int ES_, int LAYP_, int LAYQ_, int FMTP_, int FMTQ_, int NS_>
struct RingCfg {
  static constexpr int BP = BP_, BQ = BQ_, WP = WP_, WQ = WQ_, ES = ES_, NS = NS_;
  static constexpr int LAYP = LAYP_, LAYQ = LAYQ_, FMTP = FMTP_, FMTQ = FMTQ_;
  static constexpr int NW = WP * WQ, NT = NW * 64;
  static constexpr int TP = BP / WP / 32, TQ = BQ / WQ / 32;
  static constexpr int KS = ES == 2 ? 4 : 2;           // MFMA k-steps per k-tile of 128 bytes
  static constexpr int STAGE_BYTES = (BP + BQ) * 128;
  static constexpr int STAGE_LD = TP * 32 + 4;         // epilogue staging: a wavefront's slice is 32 rows of this many floats
  static constexpr int EPI_BYTES = NW * 32 * STAGE_LD * 4;
  static constexpr int LDS_BYTES = NS * STAGE_BYTES > EPI_BYTES ? NS * STAGE_BYTES : EPI_BYTES;
  static_assert(NW == 4 && NS >= 3 && NS <= TFB_MAX_RING && LDS_BYTES <= 160 * 1024, "ring");
};

template <int OFF>
__device__ __forceinline__ i32x4 ring_read128(uint32_t addr) {
  i32x4 v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
  return v;
}
template <int OFF, int ES>
__device__ __forceinline__ u32x2 ring_read_tr64(uint32_t addr) {
  u32x2 v;
  if (ES == 2) asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
  else asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
  return v;
}

// One operand's fragments of a k-tile: request() reads all of them into this object's registers, landed() ties those registers
// to the wait that precedes it, get<i, s>() is the fragment of MFMA tile i, k-step s. The layouts are FragReader's.
template <int ROWS, int NTILE, int ES, int LAY, int TILE = 32>   // TILE: as FragReader's
struct RingFrags;

template <int ROWS, int NTILE>
struct RingAddr {   // per-lane byte offsets inside a stage's operand tile
  uint32_t off[4];
};

template <int ROWS, int NTILE, int ES, int TILE>
struct RingFrags<ROWS, NTILE, ES, TFB_K_CONTIG, TILE> {
  static constexpr int KS = ES == 2 ? 4 : 2, PER = ES == 2 ? 1 : 2;   // 128-bit reads per fragment
  i32x4 v[NTILE][KS][PER];
  static __device__ __forceinline__ RingAddr<ROWS, NTILE> addr(int wave_row0, int lane) {
    const int row = wave_row0 + (lane & 31), lh = lane >> 5, f = tfb_kc_swz(row);
    RingAddr<ROWS, NTILE> a;
#pragma unroll
    for (int n = 0; n < 4; ++n) {   // n = k-step (bf16), or 2 k-step + half (fp8)
      const int chunk = ES == 2 ? 2 * n + lh : 4 * (n >> 1) + 2 * lh + (n & 1);
      a.off[n] = row * 128 + (((chunk ^ f) & 7) << 4);
    }
    return a;
  }
  __device__ __forceinline__ void request(const RingAddr<ROWS, NTILE>& a, uint32_t base) {
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      v[0][n / PER][n % PER] = ring_read128<0>(base + a.off[n]);
      if constexpr (NTILE == 2) v[1][n / PER][n % PER] = ring_read128<TILE * 128>(base + a.off[n]);
    }
  }
  __device__ __forceinline__ void landed() {
#pragma unroll
    for (int i = 0; i < NTILE; ++i)
#pragma unroll
      for (int n = 0; n < 4; ++n) asm volatile("" : "+v"(v[i][n / PER][n % PER]));
  }
  template <int i, int s>
  __device__ __forceinline__ auto get() const {
    if constexpr (ES == 2) {
      return __builtin_bit_cast(bf16x8, v[i][s][0]);
    } else {
      const i32x4 a = v[i][s][0], b = v[i][s][1];
      return i32x8{a.x, a.y, a.z, a.w, b.x, b.y, b.z, b.w};
    }
  }
};

template <int ROWS, int NTILE, int ES>
struct RingFrags<ROWS, NTILE, ES, TFB_K_STRIDED, 32> {
  static constexpr int KS = ES == 2 ? 4 : 2, PER = ES == 2 ? 2 : 4;   // 64-bit transposing reads per fragment
  static constexpr int PITCH = ROWS * ES, KSTEP = (ES == 2 ? 16 : 64) * PITCH, KQ = (ES == 2 ? 4 : 8) * PITCH;
  u32x2 v[NTILE][KS][PER];
  static __device__ __forceinline__ RingAddr<ROWS, NTILE> addr(int wave_row0, int lane) {
    const int g4 = lane >> 4, j = lane & 15;
    RingAddr<ROWS, NTILE> a;
#pragma unroll
    for (int i = 0; i < NTILE; ++i) {
      if (ES == 2) {
        const int p = wave_row0 + 32 * i + 16 * (g4 & 1) + 4 * (j & 3), k = 8 * (g4 >> 1) + (j >> 2);
        a.off[i] = k * PITCH + ((((p >> 3) ^ tfb_ks_swz<ROWS, ES>(k)) << 4) | ((p & 4) << 1));
      } else {
        const int p = wave_row0 + 32 * i + 16 * (g4 & 1) + 8 * (j & 1), k = 32 * (g4 >> 1) + (j >> 1);
        a.off[i] = k * PITCH + ((((p >> 4) ^ tfb_ks_swz<ROWS, ES>(k)) << 4) | (p & 8));
      }
    }
    return a;
  }
  template <int i, int n>
  __device__ __forceinline__ void req(const RingAddr<ROWS, NTILE>& a, uint32_t base) {
    v[i][n / PER][n % PER] = ring_read_tr64<(n / PER) * KSTEP + (n % PER) * KQ, ES>(base + a.off[i]);
    if constexpr (n + 1 < KS * PER) req<i, n + 1>(a, base);
  }
  __device__ __forceinline__ void request(const RingAddr<ROWS, NTILE>& a, uint32_t base) {
    req<0, 0>(a, base);
    if constexpr (NTILE == 2) req<1, 0>(a, base);
  }
  __device__ __forceinline__ void landed() {
#pragma unroll
    for (int i = 0; i < NTILE; ++i)
#pragma unroll
      for (int n = 0; n < KS * PER; ++n) asm volatile("" : "+v"(v[i][n / PER][n % PER]));
  }
  template <int i, int s>
  __device__ __forceinline__ auto get() const {
    if constexpr (ES == 2) {
      const u32x4 w = {v[i][s][0].x, v[i][s][0].y, v[i][s][1].x, v[i][s][1].y};
      return __builtin_bit_cast(bf16x8, w);
    } else {
      i32x8 w;
#pragma unroll
      for (int q = 0; q < 4; ++q) {
        w[2 * q] = (int)v[i][s][q].x;
        w[2 * q + 1] = (int)v[i][s][q].y;
      }
      return w;
    }
  }
};

// The MFMAs that made x stay in front of this point (they have no side effects, and would otherwise sink across barriers).
__device__ __forceinline__ void ring_pin(f32x16& x) { asm volatile("" : "+v"(x)); }

// s_waitcnt vmcnt(tiles * PER): all but the newest `tiles` k-tiles of loads have landed (tiles is wavefront-uniform)
template <int PER>
__device__ __forceinline__ void ring_wait(int tiles) {
#define TFB_RING_WAIT(n) case n: asm volatile("s_waitcnt vmcnt(%0)" ::"n"((n) * PER) : "memory"); break;
  switch (tiles) {
    TFB_RING_WAIT(1) TFB_RING_WAIT(2) TFB_RING_WAIT(3) TFB_RING_WAIT(4) TFB_RING_WAIT(5) TFB_RING_WAIT(6)
    default: asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  }
#undef TFB_RING_WAIT
}

// Workgroup `block` of the launch: one output tile (given_p >= 0: that one).
template <class Cfg, bool RANGES, class Epi>
__device__ __forceinline__ void gemm_ring_tile(GemmArgs a, const Epi& epi_in, int block, uint8_t* lds, int given_p = -1, int given_q = 0) {
  constexpr int BP = Cfg::BP, BQ = Cfg::BQ, NW = Cfg::NW, TP = Cfg::TP, TQ = Cfg::TQ, ES = Cfg::ES, NS = Cfg::NS;
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wp = wave % Cfg::WP, wq = wave / Cfg::WP;
  const int lr = lane & 31, lh = lane >> 5;
  int lid, split, tile_p, tile_q;
  [[maybe_unused]] int sym_group = 0;
  if constexpr (is_symmetric<Epi>::value) {
    static_assert(BP == BQ, "square tiles");
    // an XCD's workgroups (id & 7) take a run of consecutive tiles, so that a group's operand is read into one or two L2s only
    lid = (block & 7) * a.per + (block >> 3);
    split = 0;
    sym_group = fastdiv(lid, a.d_ntiles);
    if (sym_group >= a.rows) return;   // (the whole workgroup: the runs are of equal length)
    tile_p = lid - sym_group * a.ntiles;
    tile_q = 0;
    for (; tile_p >= a.ntp - tile_q; ++tile_q) tile_p -= a.ntp - tile_q;   // row tile_q has ntp - tile_q tiles
    tile_p += tile_q;
  } else if (given_p >= 0) {
    lid = split = 0;
    tile_p = given_p;
    tile_q = given_q;
  } else {
    gemm_tile_of(a, block, lid, split, tile_p, tile_q);
  }
  const long p0 = (long)tile_p * BP, q0 = (long)tile_q * BQ;
  int kt0 = 0;
  if (a.splits > 1) {
    kt0 = fastdiv(split * a.nkt, a.d_splits);
    a.nkt = fastdiv((split + 1) * a.nkt, a.d_splits) - kt0;
  }
  int group = 0;
  if (a.q_group) {   // (named per 128 rows of q)
    group = a.q_group[q0 >> 7];
    if (group < 0) return;  // the whole workgroup leaves before any barrier
    a.P.base += (long)group * a.p_group_stride;
  }
  if (a.k_seg) {
    group = blockIdx.y;
    const int k0 = a.k_seg[group], k1 = a.k_seg[group + 1];
    kt0 = k0 * ES / 128;
    a.nkt = (k1 - k0) * ES / 128;  // may be 0: the accumulators stay zero and are still written
  }
  if constexpr (is_symmetric<Epi>::value) {
    group = sym_group;
    a.P.base += group * a.g_stride;
    a.Q.base += group * a.g_stride;
  }
  const int nkt = a.nkt;

  typedef TileDma<BP, NW, Cfg::LAYP, ES> DP;
  typedef TileDma<BQ, NW, Cfg::LAYQ, ES> DQ;
  constexpr int NI = DP::NI + DQ::NI;   // load instructions per wavefront and k-tile
  static_assert((NS - 1) * NI < 63, "vmcnt counts to 63");
  DP dp;
  DQ dq;
  dp.init(a.P, p0, (long)kt0 * 128, wave, lane);
  dq.init(a.Q, q0, (long)kt0 * 128, wave, lane);
  auto issue = [&](int stage, int t) {
    dp.issue(lds + stage * Cfg::STAGE_BYTES, t, wave);
    dq.issue(lds + stage * Cfg::STAGE_BYTES + BP * 128, t, wave);
  };
#pragma unroll
  for (int t = 0; t < NS; ++t)
    if (t < nkt) issue(t, t);

  const Epi epi = epi_prepare(epi_for_group(epi_in, group));
  constexpr bool kFar = partner_of<Epi>::value == 64;
  static_assert(!kFar || (BP == 128 && Cfg::WP == 2 && Cfg::LAYP == TFB_K_CONTIG), "whole heads of 128");
  typedef RingFrags<BP, TP, ES, Cfg::LAYP, kFar ? 64 : 32> FP;
  typedef RingFrags<BQ, TQ, ES, Cfg::LAYQ> FQ;
  const auto ap = FP::addr(wp * (kFar ? 32 : TP * 32), lane);
  const auto aq = FQ::addr(wq * (TQ * 32), lane);
  const uint32_t lds0 = (uint32_t)(uintptr_t)(tfb_lds_void_t*)lds;
  FP fp[2];
  FQ fq[2];
  auto request = [&](int set, int stage) {
    const uint32_t b = lds0 + stage * Cfg::STAGE_BYTES;
    fp[set].request(ap, b);
    fq[set].request(aq, b + BP * 128);
  };

  f32x16 acc[TP][TQ];
#pragma unroll
  for (int i = 0; i < TP; ++i)
#pragma unroll
    for (int j = 0; j < TQ; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;

  // symmetric products: the second half of every k-tile has sums of its own, as in gemm_sym.hpp
  constexpr bool HALVES = is_symmetric<Epi>::value;
  [[maybe_unused]] f32x16 upper[HALVES ? TP : 1][HALVES ? TQ : 1];
  if constexpr (HALVES) {
#pragma unroll
    for (int i = 0; i < TP; ++i)
#pragma unroll
      for (int j = 0; j < TQ; ++j) upper[i][j] = acc[i][j];
  }

  // a.ranges k ranges [z nkt / Z, (z + 1) nkt / Z), as a k-split cuts them: total = range 0 + range 1 + ...
  [[maybe_unused]] f32x16 total[RANGES ? TP : 1][RANGES ? TQ : 1];
  [[maybe_unused]] int range = 1, range_end = RANGES ? fastdiv(nkt, a.d_ranges) : 0;
  auto fold = [&]() {
#pragma unroll
    for (int i = 0; i < TP; ++i)
#pragma unroll
      for (int j = 0; j < TQ; ++j) {
        total[i][j] = range == 1 ? acc[i][j] : total[i][j] + acc[i][j];
#pragma unroll
        for (int e = 0; e < 16; ++e) acc[i][j][e] = 0.f;
      }
    ++range;
    range_end = fastdiv(range * nkt, a.d_ranges);
  };

  // the staged epilogue's chunk of pass k: row and first column inside the wavefront's 32-row slice
  constexpr bool kPrefetch = has_prefetch<Epi>::value && !has_tile_epilogue<Epi>::value;
  constexpr int CPR = TP * 4, NK = 32 * CPR / 64;
  auto chunk_row = [&](int k) { return 2 * (((lane >> 3) + k * 8) / (CPR / 4)) + ((lane >> 2) & 1); };
  auto chunk_col = [&](int k) { return (4 * (((lane >> 3) + k * 8) % (CPR / 4)) + (lane & 3)) * 8; };
  const int pw = wp * (TP * 32), qw = wq * (TQ * 32);  // wavefront's origin inside the tile
  [[maybe_unused]] typename prefetch_type<Epi>::type pre[TQ][NK];

  // k-step s of a set: every operand pair's MFMA
  auto mfmas = [&](int set, auto s_) {
    constexpr int s = decltype(s_)::value;
    auto one = [&](auto i_, auto j_) {
      constexpr int i = decltype(i_)::value, j = decltype(j_)::value;
      auto& c = [&]() -> f32x16& {
        if constexpr (HALVES && 2 * s >= Cfg::KS) return upper[i][j];
        else return acc[i][j];
      }();
      c = mfma32<ES, Cfg::FMTP, Cfg::FMTQ>(fp[set].template get<i, s>(), fq[set].template get<j, s>(), c);
    };
    using N0 = std::integral_constant<int, 0>;
    using N1 = std::integral_constant<int, 1>;
    one(N0{}, N0{});
    if constexpr (TQ == 2) one(N0{}, N1{});
    if constexpr (TP == 2) one(N1{}, N0{});
    if constexpr (TP == 2 && TQ == 2) one(N1{}, N1{});
  };

  int stage = 0;   // of the k-tile whose fragments were requested last
  // k-tile t, whose fragments were requested into `set`: the next k-tile's are requested, its own multiplied. full_: there
  // is a k-tile t + NS to load (the loop's body then has no branches)
  auto step = [&](int set, int t, auto full_) {
    constexpr bool full = decltype(full_)::value;
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
    fp[set].landed();
    fq[set].landed();
    if (full || t + 1 < nkt) {
      const int left = nkt - 2 - t;
      ring_wait<NI>(full || left > NS - 2 ? NS - 2 : left);
      // behind this barrier every wavefront has k-tile t in registers (its stage is free) and its share of t + 1 in LDS
      __builtin_amdgcn_sched_barrier(0);
      asm volatile("s_barrier" ::: "memory");
      __builtin_amdgcn_sched_barrier(0);
      if (full || t + NS < nkt) issue(stage, t + NS);
      stage = stage + 1 == NS ? 0 : stage + 1;
      request(set ^ 1, stage);
    }
    if constexpr (RANGES)
      if (t == range_end) fold();
    mfmas(set, std::integral_constant<int, 0>{});
    mfmas(set, std::integral_constant<int, 1>{});
    if constexpr (Cfg::KS == 4) {
      mfmas(set, std::integral_constant<int, 2>{});
      mfmas(set, std::integral_constant<int, 3>{});
    }
#pragma unroll
    for (int i = 0; i < TP; ++i)
#pragma unroll
      for (int j = 0; j < TQ; ++j) {
        ring_pin(acc[i][j]);
        if constexpr (HALVES) ring_pin(upper[i][j]);
      }
  };

  if (nkt > 0) {
    ring_wait<NI>(nkt - 1 < NS - 1 ? nkt - 1 : NS - 1);
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("s_barrier" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
    request(0, 0);
  }
  if constexpr (kPrefetch) {   // the epilogue's own operands fly under the k-loop
#pragma unroll
    for (int j = 0; j < TQ; ++j)
#pragma unroll
      for (int k = 0; k < NK; ++k) pre[j][k] = epi.prefetch((int)p0 + tfb_slice_col<Epi>(wp, TP * 32, chunk_col(k)), a.q_off + (int)q0 + qw + j * 32 + chunk_row(k));
  }
  int t = 0;
  for (; t + 1 + NS < nkt; t += 2) {
    step(0, t, std::true_type{});
    step(1, t + 1, std::true_type{});
  }
  for (; t < nkt; t += 2) {
    step(0, t, std::false_type{});
    if (t + 1 < nkt) step(1, t + 1, std::false_type{});
  }
  // (nothing is on its way into the fragments' registers here, on no path: the check of the built code follows them all)
  asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");
#pragma unroll
  for (int set = 0; set < 2; ++set) {
    fp[set].landed();
    fq[set].landed();
  }
  if constexpr (RANGES) {
    if (range > 1) {
#pragma unroll
      for (int i = 0; i < TP; ++i)
#pragma unroll
        for (int j = 0; j < TQ; ++j) acc[i][j] = total[i][j] + acc[i][j];
    }
  }
  if constexpr (HALVES) {
#pragma unroll
    for (int i = 0; i < TP; ++i)
#pragma unroll
      for (int j = 0; j < TQ; ++j) acc[i][j] = acc[i][j] + upper[i][j];
  }
  __syncthreads();

  if constexpr (has_tile_epilogue<Epi>::value) {
    epi.tile(acc, (int)p0 + pw, a.q_off + (int)q0 + qw, lr, lh, lid, split);
  } else {
    // 32 output rows at a time through the wavefront's own LDS slice, then 8-element chunks, a row's on consecutive lanes
    constexpr int SLD = Cfg::STAGE_LD;
    float* stg = (float*)lds + wave * (32 * SLD);
    typedef MirrorBlock<TP * 32> Mirror;
    static_assert(!is_symmetric<Epi>::value || Cfg::EPI_BYTES + NW * (Mirror::BYTES + Mirror::OUT_BYTES) <= Cfg::LDS_BYTES, "mirror slices");
    [[maybe_unused]] uint8_t* mirror = lds + Cfg::EPI_BYTES + wave * (Mirror::BYTES + Mirror::OUT_BYTES);
#pragma unroll
    for (int j = 0; j < TQ; ++j) {
#pragma unroll
      for (int i = 0; i < TP; ++i)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const f32x4 v = {acc[i][j][jj * 4 + 0], acc[i][j][jj * 4 + 1], acc[i][j][jj * 4 + 2], acc[i][j][jj * 4 + 3]};
          *(f32x4*)(stg + lr * SLD + i * 32 + jj * 8 + lh * 4) = v;
        }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int k = 0; k < NK; ++k) {
        const int row = chunk_row(k), pc = chunk_col(k);
        const int p = (int)p0 + tfb_slice_col<Epi>(wp, TP * 32, pc), q = a.q_off + (int)q0 + qw + j * 32 + row;
        const f32x4 lo = *(const f32x4*)(stg + row * SLD + pc), hi = *(const f32x4*)(stg + row * SLD + pc + 4);
        const float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        if constexpr (is_symmetric<Epi>::value) {
          u32x4 w;
          if constexpr (kPrefetch) w = epi.value(v, pre[j][k]);
          else w = epi.value(v);
          *(u32x4*)(epi.out + (long)q * epi.ld + p) = w;
          if (tile_p != tile_q) Mirror::put(mirror, row, pc, w);
        } else if constexpr (partner_of<Epi>::value != 0) {
          static_assert(TP == 2, "partner epilogue: 64 staged columns per wavefront");
          const f32x4 plo = *(const f32x4*)(stg + row * SLD + (pc ^ 32)), phi = *(const f32x4*)(stg + row * SLD + (pc ^ 32) + 4);
          const float vp[8] = {plo[0], plo[1], plo[2], plo[3], phi[0], phi[1], phi[2], phi[3]};
          if constexpr (kPrefetch) epi(p, q, v, vp, pre[j][k], split);
          else epi(p, q, v, vp, split);
        } else if constexpr (kPrefetch) {
          epi(p, q, v, pre[j][k], split);
        } else {
          epi(p, q, v, split);
        }
      }
      __builtin_amdgcn_wave_barrier();
      if constexpr (is_symmetric<Epi>::value) {
        if (tile_p != tile_q) Mirror::store(mirror, mirror + Mirror::BYTES, epi.out + ((long)p0 + pw) * epi.ld + q0 + qw + j * 32, epi.ld, lane);
      }
    }
  }
}

template <class Cfg, bool RANGES, class Epi>
__global__ __launch_bounds__(Cfg::NT, 2) void gemm_ring_kernel(GemmArgs a, Epi epi_in) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[Cfg::LDS_BYTES];
  gemm_ring_tile<Cfg, RANGES>(a, epi_in, blockIdx.x, lds);
}

// ranges > 1: the k ranges summed inside the workgroup (at most nkt of them; not with a k_seg)
template <class Cfg>
static int gemm_ring_args(GemmArgs& a, int splits, int ranges) {
  const int st = gemm_map_args<Cfg>(a, splits);
  if (st != TFB_OK) return st;
  a.slots = 0;
  a.sleeps = 0;
  if (ranges > 1 && (splits > 1 || ranges > a.nkt)) return TFB_ERR_SHAPE;
  a.ranges = ranges;
  a.d_ranges = fastdiv_make(ranges);
  return TFB_OK;
}
template <class Cfg, class Epi>
static int gemm_ring_launch_args(GemmArgs a, int groups_y, int splits, int ranges, Epi epi, hipStream_t stream) {
  const int st = gemm_ring_args<Cfg>(a, splits, ranges);
  if (st != TFB_OK) return st;
  const dim3 grid(a.ntiles * splits, groups_y, 1);
  if constexpr (has_ranges<Epi>::value) {
    if (ranges > 1) {
      hipLaunchKernelGGL((gemm_ring_kernel<Cfg, true, Epi>), grid, dim3(Cfg::NT), 0, stream, a, epi);
      TFB_LAUNCH_CHECK();
      return TFB_OK;
    }
  }
  if (ranges > 1) return TFB_ERR_ARG;
  hipLaunchKernelGGL((gemm_ring_kernel<Cfg, false, Epi>), grid, dim3(Cfg::NT), 0, stream, a, epi);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}

// Which ring tile a launch of np x nq outputs (times `groups` equal ones) and nkt k-tiles takes: 1 = 64 x 64, 2 = 128 (p) x 64 (q),
// 0 = none (the 128 x 128 core or the persistent kernel). A CU moves some 30 bytes per clock into LDS whatever the tile, so the
// time is the bytes of the CU with the most tiles: 64 x 64 while every tile has a CU of its own, then 128 x 64 (3/4 of the bytes per
// output) while no CU has more than two (k-strided operands, which cost the core more: two and a quarter); beyond, the core's two
// workgroups per CU hide as much. Measured standalone, core -> ring (us): bf16 256 x 768 x 768 10.6 -> 4.9, 2048 x 768 x 768
// 11.0 -> 6.7, 2048 x 768 x 2304 20.9 -> 13.3, 4096 x 768 x 768 11.4 -> 10.4, 2048 x 2304 x 768 14.5 -> 15.0 (576 tiles of
// 128 x 64: beyond the line); fp8 1024 x 768 x 3072 18.7 -> 7.2, 2048 x 768 x 3072 18.8 -> 10.0, 4096 x 1024 x 4096 25.7 -> 20.4;
// token contractions 2304 x 768 over 2048 24.2 -> 12.5, 768 x 768 over 1024 16.0 -> 6.2, fp8 3072 x 768 over 2048 14.7 -> 11.9.
// From 96 k-tiles on the k-split forms of the other kernels are as good or better.
static inline int gemm_ring_pick(long np, long nq, long nkt, bool strided, long groups = 1) {
  if (nkt <= 0 || nkt > 96) return 0;
  const long cus = tfb_resident_slots(1), t64 = (np / 64) * (nq / 64) * groups;
  if (t64 <= cus) return 1;
  return 2 * t64 <= (strided ? 9 : 8) * cus ? 2 : 0;
}

// A stack of `groups` symmetric N x N products of one operand with itself (N a multiple of 128) on 64 x 64 tiles: gemm_sym.hpp has the rule.
template <class Epi, int ES, int LAY>
static int gemm_ring_symmetric(GemmOperand X, long g_stride, int N, int nkt, int groups, Epi e, hipStream_t s) {
  GemmArgs a = {};
  a.P = X;
  a.Q = X;
  a.np = N;
  a.nq = N;
  a.nkt = nkt;
  a.g_stride = g_stride;
  a.ntp = N / 64;
  using Cfg = RingCfg<64, 64, 2, 2, ES, LAY, LAY, 0, 0, 4>;
  const int st = gemm_map_args<Cfg>(a, 1);
  if (st != TFB_OK) return st;
  a.ntiles = a.ntp * (a.ntp + 1) / 2;
  a.d_ntiles = fastdiv_make(a.ntiles);
  a.rows = groups;
  if ((long)a.ntiles * groups > 0x7ffffff0L / 8) return TFB_ERR_SHAPE;
  a.per = (a.ntiles * groups + 7) / 8;
  hipLaunchKernelGGL((gemm_ring_kernel<Cfg, false, Epi>), dim3(8 * a.per), dim3(256), 0, s, a, e);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}

template <class Epi, int ES, int LAYP, int LAYQ, int FMTP, int FMTQ>
static int gemm_ring_launch(int pick, GemmArgs a, int groups_y, int splits, Epi e, hipStream_t s, int ranges = 1, int q_off = 0) {
  a.q_off = q_off;
  if constexpr (partner_of<Epi>::value == 0 && !has_tile_epilogue<Epi>::value) {   // (those take 64 columns of p per wavefront)
    if (pick == 1) {
      a.ntp = a.np / 64;
      return gemm_ring_launch_args<RingCfg<64, 64, 2, 2, ES, LAYP, LAYQ, FMTP, FMTQ, 4>>(a, groups_y, splits, ranges, e, s);
    }
  }
  a.ntp = a.np / 128;
  return gemm_ring_launch_args<RingCfg<128, 64, 2, 2, ES, LAYP, LAYQ, FMTP, FMTQ, 3>>(a, groups_y, splits, ranges, e, s);
}

// A dense launch through the ring where gemm_ring_pick takes it: true, with its status in st.
template <int ES, int LAYP, int LAYQ, int FMTP, int FMTQ, class Epi>
static bool gemm_ring_try(GemmOperand P, GemmOperand Q, int np, int nq, long kbytes, Epi e, hipStream_t s, int& st, int ranges = 1) {
  const int pick = gemm_ring_pick(np, nq, kbytes / 128, LAYP == TFB_K_STRIDED && LAYQ == TFB_K_STRIDED);
  if (!pick || np % 128 || nq % 128 || kbytes % 128) return false;
  GemmArgs a = {};
  a.P = P;
  a.Q = Q;
  a.np = np;
  a.nq = nq;
  a.nkt = (int)(kbytes / 128);
  st = gemm_ring_launch<Epi, ES, LAYP, LAYQ, FMTP, FMTQ>(pick, a, 1, 1, e, s, ranges);
  return true;
}

// A dense launch through the persistent kernel where gemm_pp_shape gives it a tile (all but the last 128 rows of q, it may be: those go
// through the ring: 9600 x 3072 x 1024 in bf16 79 -> 62 us): true, with its status in st. heavy: the epilogue is heavy there.
template <int ES, int LAYP, int LAYQ, int FMTP, int FMTQ, class Epi>
static bool gemm_pp_try(GemmOperand P, GemmOperand Q, int np, int nq, long kbytes, bool heavy, Epi e, hipStream_t s, int& st) {
  constexpr bool rotation = partner_of<Epi>::value != 0, narrow_ok = LAYQ == TFB_K_CONTIG && !rotation;
  const int shape = gemm_pp_shape(np, nq, kbytes, heavy && !rotation, narrow_ok, rotation ? 1.04 : 1.0);
  if (shape < 0) return false;
  if constexpr (narrow_ok) {
    if (shape == TFB_PP_192x256) st = gemm_pp_launch_lay<ES, FMTP, FMTQ, LAYP, LAYQ, TFB_PP_192x256>(P, Q, np, nq, kbytes, 1, e, s);
    if (shape == TFB_PP_256x192) st = gemm_pp_launch_lay<ES, FMTP, FMTQ, LAYP, LAYQ, TFB_PP_256x192>(P, Q, np, nq, kbytes, 1, e, s);
    if (shape != TFB_PP_256x256) return true;
  }
  const int rest = nq % 256, main = nq - rest;
  st = gemm_pp_launch_lay<ES, FMTP, FMTQ, LAYP, LAYQ>(P, Q, np, main, kbytes, 1, e, s);
  if (st != TFB_OK || !rest) return true;
  GemmArgs a = {};
  a.P = P;
  a.Q = GemmOperand{Q.base + (LAYQ == TFB_K_CONTIG ? main * Q.ld : (long)main * ES), Q.ld};
  a.np = np;
  a.nq = rest;
  a.nkt = (int)(kbytes / 128);
  st = gemm_ring_launch<Epi, ES, LAYP, LAYQ, FMTP, FMTQ>(128L * np <= 4096L * tfb_resident_slots(1) ? 1 : 2, a, 1, 1, e, s, 1, main);
  return true;
}

// What the persistent kernel leaves of a grouped product over rows (RowItems): its last output tiles as 128 x 64 ones, eight workgroups each.
template <class Cfg, class Epi>
__global__ __launch_bounds__(Cfg::NT, 2) void gemm_ring_rest_kernel(GemmArgs a, Epi epi_in, int row_tiles, int ncol, FastDiv d_ncol, int nwg) {
  __shared__ __attribute__((aligned(1024))) uint8_t lds[Cfg::LDS_BYTES];
  static_assert(Cfg::BP == 128 && Cfg::BQ == 64, "eight tiles of 256 x 256");
  const int lane = threadIdx.x & 63, sub = blockIdx.x & 7;
  RowItems ri;
  ri.init(a.q_group, row_tiles, ncol, nwg, lane);
  const int w = ri.taken + (int)(blockIdx.x >> 3);
  if (w >= ri.total) return;  // (the whole workgroup, as below)
  const int k = fastdiv(w, d_ncol), t = __builtin_amdgcn_readfirstlane(ri.tile(k, lane));
  if (sub >= 4 && (t + 1 >= row_tiles || a.q_group[t + 1] != a.q_group[t])) return;
  gemm_ring_tile<Cfg, false>(a, epi_in, 0, lds, 2 * (w - k * ncol) + (sub & 1), 2 * t + (sub >> 1));
}
template <int FMTP, int FMTQ, class Epi>
static int gemm_ring_rest(GemmArgs a, Epi e, hipStream_t s) {
  using Cfg = RingCfg<128, 64, 2, 2, 1, TFB_K_CONTIG, TFB_K_CONTIG, FMTP, FMTQ, 3>;
  a.ntp = a.np / 128;
  a.q_off = 0;
  const int row_tiles = a.nq / 128, ncol = a.np / 256, nwg = gemm_pp_rows_wgs();
  const int st = gemm_ring_args<Cfg>(a, 1, 1);
  if (st != TFB_OK) return st;
  const long most = std::min((long)row_tiles * ncol, 3L * nwg / 10 + 1);
  hipLaunchKernelGGL((gemm_ring_rest_kernel<Cfg, Epi>), dim3((unsigned)(8 * most)), dim3(Cfg::NT), 0, s, a, e, row_tiles, ncol, fastdiv_make(ncol), nwg);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}

// ---- several independent contractions in one launch ------------------------------------------------------------------
// What bounds a ring launch is the rate at which a CU's loads go into LDS (some 100 KB a microsecond, whatever the tile or the number
// of stages; the loads alone take 12.5 of the 13.9 us of a 2048 x 768 x 2304 launch), and a launch of fewer tiles than CUs leaves the
// others idle for its whole length. The gradients of one layer - the input's and the weights' - are independent of each other, so they
// run as jobs of one launch: the tiles of the second start where the first leaves room, and a launch's fixed 3 - 4 us are paid once.
// The same tiles, the same sums as in launches of their own.
template <int LAYP_, int LAYQ_, int ES_, int FMTP_, int FMTQ_, bool RANGES_, class Epi_>
struct RingJob {
  typedef Epi_ Epi;
  static constexpr bool RANGES = RANGES_;
  template <int BP, int NS>
  using Cfg = RingCfg<BP, 64, 2, 2, ES_, LAYP_, LAYQ_, FMTP_, FMTQ_, NS>;
  typedef Cfg<64, 4> Small;
  typedef Cfg<128, 3> Large;
  GemmArgs a = {};
  Epi e;
  int ranges = 1;
  RingJob(GemmOperand P, GemmOperand Q, int np, int nq, long kbytes, Epi e_, int ranges_ = 1) : e(e_), ranges(ranges_) {
    a.P = P;
    a.Q = Q;
    a.np = np;
    a.nq = nq;
    a.nkt = (int)(kbytes / 128);
  }
  double bytes() const { return (double)(a.np / 128) * (a.nq / 64) * a.nkt * 24576; }   // through LDS, in tiles of 128 x 64
};
template <class Cfg_, class Job>
struct RingPart {
  typedef Cfg_ Cfg;
  GemmArgs a;
  typename Job::Epi e;
  int first, blocks;   // its workgroups; a multiple of 8, so that an id keeps its XCD
};
struct RingNoJob {
  typedef RingNoJob Small, Large, Epi;
  static constexpr int LDS_BYTES = 0;
  static constexpr bool RANGES = false;
  GemmArgs a = {};
  double bytes() const { return 0; }
};

template <class J, class Part>
__device__ __forceinline__ void gemm_ring_part(const Part& p, uint8_t* lds) {
  const int block = (int)blockIdx.x - p.first;
  if (block >= 0 && block < p.a.ntiles) gemm_ring_tile<typename Part::Cfg, J::RANGES>(p.a, p.e, block, lds);
}
template <class J0, class J1, class J2, class P0, class P1, class P2>
__global__ __launch_bounds__(256, 2) void gemm_ring_jobs_kernel(P0 p0, P1 p1, P2 p2) {
  constexpr int B01 = P0::Cfg::LDS_BYTES > P1::Cfg::LDS_BYTES ? P0::Cfg::LDS_BYTES : P1::Cfg::LDS_BYTES;
  __shared__ __attribute__((aligned(1024))) uint8_t lds[B01 > P2::Cfg::LDS_BYTES ? B01 : P2::Cfg::LDS_BYTES];
  gemm_ring_part<J0>(p0, lds);
  gemm_ring_part<J1>(p1, lds);
  if constexpr (!std::is_same<J2, RingNoJob>::value) gemm_ring_part<J2>(p2, lds);
}

template <class Cfg, class Job>
static int gemm_ring_make(const Job& j, RingPart<Cfg, Job>& p, int& blocks, long& tile) {
  p.first = p.blocks = 0;
  if constexpr (std::is_same<Job, RingNoJob>::value) {
    return TFB_OK;
  } else {
    p.a = j.a;
    p.e = j.e;
    p.a.ntp = j.a.np / Cfg::BP;
    const int st = gemm_ring_args<Cfg>(p.a, 1, j.ranges);
    p.blocks = (p.a.ntiles + 7) & ~7;
    blocks += p.blocks;
    tile = (long)j.a.nkt * Cfg::STAGE_BYTES;
    return st;
  }
}
template <class C0, class C1, class C2, class J0, class J1, class J2>
static int gemm_ring_jobs_launch(const J0& j0, const J1& j1, const J2& j2, hipStream_t s) {
  RingPart<C0, J0> p0 = {};
  RingPart<C1, J1> p1 = {};
  RingPart<C2, J2> p2 = {};
  int n = 0;
  long t0 = 0, t1 = 0, t2 = 0;   // bytes of a tile: the longest tiles start first
  int st = gemm_ring_make(j0, p0, n, t0);
  if (st == TFB_OK) st = gemm_ring_make(j1, p1, n, t1);
  if (st == TFB_OK) st = gemm_ring_make(j2, p2, n, t2);
  if (st != TFB_OK) return st;
  p0.first = (t1 > t0 ? p1.blocks : 0) + (t2 > t0 ? p2.blocks : 0);
  p1.first = (t0 >= t1 ? p0.blocks : 0) + (t2 > t1 ? p2.blocks : 0);
  p2.first = (t0 >= t2 ? p0.blocks : 0) + (t1 >= t2 ? p1.blocks : 0);
  hipLaunchKernelGGL((gemm_ring_jobs_kernel<J0, J1, J2, RingPart<C0, J0>, RingPart<C1, J1>, RingPart<C2, J2>>), dim3(n), dim3(256), 0, s, p0, p1,
                     p2);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}
// Two jobs, or three of which the last two have the same tiles. 64 x 64 tiles for a job whose 128 x 64 tile would be longer than what a
// CU has to do on average (the output projection's weight gradient of 2048 tokens: 72 such tiles of 32 k-tiles).
template <class J0, class J1, class J2 = RingNoJob>
static int gemm_ring_jobs(const J0& j0, const J1& j1, hipStream_t s, const J2& j2 = {}) {
  const double most = 1.2 * (j0.bytes() + j1.bytes() + j2.bytes()) / tfb_resident_slots(1);
  const bool s0 = j0.a.nkt * 24576.0 > most, s1 = j1.a.nkt * 24576.0 > most;
  typedef typename J0::Small S0;
  typedef typename J0::Large L0;
  typedef typename J1::Small S1;
  typedef typename J1::Large L1;
  typedef typename J2::Small S2;
  typedef typename J2::Large L2;
  if (s0) return s1 ? gemm_ring_jobs_launch<S0, S1, S2>(j0, j1, j2, s) : gemm_ring_jobs_launch<S0, L1, L2>(j0, j1, j2, s);
  return s1 ? gemm_ring_jobs_launch<L0, S1, S2>(j0, j1, j2, s) : gemm_ring_jobs_launch<L0, L1, L2>(j0, j1, j2, s);
}
