// Weight-stationary fp8 GEMM for a contraction of 768 or 1024 bytes: D[q][p] = sum_k Q[q][k] P[p][k], P = a weight layout [np][K]
// (rows = the output's contiguous dimension), Q = token-major fp8 activations [nq][K]. For the MLP's up-projection and
// its dH GEMM (32768 x 3072 outputs from K = d_model = 768), whose cost on the tiled kernels is not the matrix pipe but
// the CU's vector-memory path: a 128 x 128 tile fetches 196 KB of operands for 48 KB of output, and ~24 bytes per clock
// and CU is what that path sustains.
//
// Here a workgroup (8 wavefronts, one per CU) keeps a PANEL of 256 weight rows in registers for its whole life - a
// wavefront holds 32 rows x K bytes as the twelve (sixteen) A fragments of v_mfma_scale_f32_32x32x64_f8f6f4 (96 or 128 registers) - and
// only the tokens stream: 64-token tiles (48 KB) through a two-stage LDS ring by global_load_lds_dwordx4, every
// wavefront reading all of a tile as B fragments. Operand traffic per output falls by four. With K = 1024 two stages of 64 tokens and
// the staging would be 192 KB of LDS: tiles of 32 tokens, four stages, asked for three tiles ahead (two stages, a tile ahead: 16384 x
// 4096 outputs up / dH 92 / 108 us instead of 87 / 99).
//
// The wavefronts form two groups (0-3, 4-7: one of each on every SIMD) that alternate roles in phases separated by one
// s_barrier: while one group multiplies tile t (24 or 16 MFMAs per wavefront) and leaves its fp32 accumulators in LDS, the
// other turns its previous tile's accumulators into outputs (the epilogue's vector work, loads and stores), which is the longer of the
// two: a wavefront alone issues an instruction every five to six cycles (accumulators staged by the finishing group instead, in 32 KB that
// the groups share: 89 -> 104 us at 32768 x 3072 x 768). The
// accumulators pass through LDS so that a wavefront pair (64 consecutive p) can finish whole 128-byte rows: after the
// phase's barrier wavefront 2m takes the first half of the pair's tokens x 64 block, wavefront 2m + 1 the other, a lane
// 8 consecutive p of one token - the operator()(p, q, v[8] [, prefetched], split) protocol of the 128 x 128 kernel's
// epilogues, which run here unchanged and see the same sums in the same order (k ascending in steps of 64).
//
// Work: XCD x (= workgroup & 7) owns an eighth of the token tiles (one more or less) and walks all panels over it in panel-major order, cut into
// equal runs for its workgroups (C4: 64 tiles x 12 panels = 768 steps = 24 per workgroup), so the slice (3 MB of fp8)
// stays in that XCD's L2 while the panels pass over it. A run that crosses a panel border reloads its registers once.
#pragma once
#include "gemm_pp.hpp"

struct Ws8Args {
  GemmOperand P, Q;
  int panels;
  int tq, more;   // token tiles per XCD; the first `more` XCDs have one more
  int per_wg;     // steps per workgroup (a step = one token tile under one panel; an XCD's steps in panel-major order)
  FastDiv d_tq, d_tq1;       // by tq, by tq + 1
  const int* row_group;      // kRows: the group of each 128 rows of Q (-1: nobody's), whose weights lie p_group_stride bytes apart
  long p_group_stride;
  int row_tiles;             // entries of row_group
};
// kRows. An XCD's tiles are a range of row_group's entries; the ranges have about the same cost, a tile of 128 rows counting WS8_TILE and a
// group's first one WS8_START more (the weights of another group are other registers to load: with eight experts of which six have three tiles
// each, all of them in the last XCD's eighth, 32768 x 2816 x 1024 182 / 188 us up / dH with equal numbers of tiles, 151 / 161 so; 6 and 9 for
// WS8_START 158 / 170 and 161 / 171). A tile that nobody has, in front of the last one that somebody has, counts like another: it takes as many
// steps, and no range is then longer than a wavefront keeps. Only the device knows the groups' loads: every wavefront reads the table for itself.
constexpr int WS8_TILE = 2, WS8_START = 4, WS8_CHUNKS = 13;   // WS8_CHUNKS: of 64 entries
constexpr long WS8_ROWS_MAX = 128L * 800;   // of 800 entries an XCD's range has 244 at most; a wavefront keeps 256
struct Ws8Range {
  int first, count;
  __device__ __forceinline__ void init(const int* group, int tiles, int x, int lane) {
    int g[WS8_CHUNKS];
#pragma unroll
    for (int c = 0; c < WS8_CHUNKS; ++c) g[c] = 64 * c + lane < tiles ? group[64 * c + lane] : -1;
    int end = 0;   // behind the last tile that somebody has
#pragma unroll
    for (int c = 0; c < WS8_CHUNKS; ++c) {
      const unsigned long long live = __ballot(g[c] >= 0);
      if (live) end = 64 * c + 64 - __builtin_clzll(live);
    }
    int cost[WS8_CHUNKS], starts = 0, before = -1;   // cost: of the entries in front of this lane's
    const unsigned long long lower = lane ? ~0ull >> (64 - lane) : 0;
#pragma unroll
    for (int c = 0; c < WS8_CHUNKS; ++c) {
      const int up = __shfl_up(g[c], 1, 64), gp = lane ? up : before;
      const unsigned long long start = __ballot(g[c] >= 0 && (g[c] != gp || 64 * c + lane == 0));
      cost[c] = WS8_TILE * (64 * c + lane) + WS8_START * (starts + __builtin_popcountll(start & lower));
      starts += __builtin_popcountll(start);
      before = __builtin_amdgcn_readlane(g[c], 63);
    }
    const int total = WS8_TILE * end + WS8_START * starts;
    int b[2];
#pragma unroll
    for (int e = 0; e < 2; ++e) {
      const int share = (total * (x + e) + 7) >> 3;
      b[e] = 0;
#pragma unroll
      for (int c = 0; c < WS8_CHUNKS; ++c) b[e] += __builtin_popcountll(__ballot(64 * c + lane < end && cost[c] < share));
    }
    first = b[0];
    count = b[1] - b[0];
  }
};

#ifndef TFB_WS8
#define TFB_WS8 1  // 0: these GEMMs stay on the tiled kernels
#endif
// a k-step's fragments are there (AFTER: reads issued behind them)
template <int NA, int AFTER>
__device__ __forceinline__ void ws8_landed(i32x4 (&b)[2 * NA]) {
  if constexpr (NA == 2) asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(b[0]), "+v"(b[1]), "+v"(b[2]), "+v"(b[3]) : "n"(AFTER));
  else asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(b[0]), "+v"(b[1]) : "n"(AFTER));
}
template <int I, int N, class F>
__device__ __forceinline__ void ws8_unroll(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    ws8_unroll<I + 1, N>(f);
  }
}

// An epilogue may take an element's place in its outputs (place(p, q), linear in q) instead of its coordinates: put(place, v [, prefetched]).
// A product of 64 bits for every row of a lane is a large part of what it does.
template <class T, class = void>
struct has_place : std::false_type {};
template <class T>
struct has_place<T, std::void_t<decltype(std::declval<const T&>().place(0, 0))>> : std::true_type {};

// NK: the contraction in k-tiles of 128 bytes
template <int NK, int FMTP, int FMTQ, class Epi>
__global__ __launch_bounds__(512, 2) void gemm_ws8_kernel(Ws8Args a, Epi epi_in) {
  constexpr int TT = NK <= 6 ? 64 : 32, NS = NK <= 6 ? 2 : 4;  // tokens per tile, stages
  constexpr int NA = TT / 32, KS = 2 * NK;                     // accumulators, k-steps
  constexpr int ND = TT == 64 ? NK : NK / 2;  // a wavefront's load instructions for a tile
  constexpr int NP = TT / 16;                                       // passes of a wavefront's epilogue (8 tokens each)
  constexpr int STAGE = NK * TT * 128;  // TT tokens, as NK k-tiles of [TT rows][128 bytes]
  __shared__ __attribute__((aligned(1024))) uint8_t ring[NS * STAGE];
  __shared__ __attribute__((aligned(1024))) uint8_t stg_all[4 * TT * 256];  // per wavefront pair: TT tokens x 64 p fp32
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int grp = wave >> 2;  // wavefronts w and w + 4 share a SIMD
  const int lr = lane & 31, lh = lane >> 5;

  const int x = blockIdx.x & 7, wi = blockIdx.x >> 3;
  constexpr bool kRows = has_rows<Epi>::value;
  [[maybe_unused]] Ws8Range range = {};
  if constexpr (kRows) range.init(a.row_group, a.row_tiles, x, lane);
  constexpr int PER = 128 / TT;
  const int tq = kRows ? PER * range.count : a.tq + (x < a.more ? 1 : 0);
  const int tile0 = kRows ? PER * range.first : x * a.tq + (x < a.more ? x : a.more);
  const int per_wg = kRows ? (a.panels * tq + (gridDim.x >> 3) - 1) / (int)(gridDim.x >> 3) : a.per_wg;
  const int s0 = wi * per_wg;
  int T = a.panels * tq - s0;
  if (T > per_wg) T = per_wg;
  if (T <= 0) return;  // (whole workgroup, before any barrier)
  [[maybe_unused]] int rg[4];   // the groups of this XCD's tiles: entry i in lane i & 63 of rg[i >> 6]
  [[maybe_unused]] float inv_tq = 0.f;
  if constexpr (kRows) {
    inv_tq = 1.0f / (float)tq;
#pragma unroll
    for (int i = 0; i < 4; ++i) rg[i] = 64 * i + lane < range.count ? a.row_group[range.first + 64 * i + lane] : -1;
    asm volatile("s_waitcnt vmcnt(0)" : "+v"(rg[0]), "+v"(rg[1]), "+v"(rg[2]), "+v"(rg[3]));
  }
  auto group_at = [&](long q0) {
    const int i = (int)(q0 >> 7) - range.first, l = i & 63;
    const int v[4] = {__builtin_amdgcn_readlane(rg[0], l), __builtin_amdgcn_readlane(rg[1], l), __builtin_amdgcn_readlane(rg[2], l),
                      __builtin_amdgcn_readlane(rg[3], l)};
    return i < 128 ? (i < 64 ? v[0] : v[1]) : (i < 192 ? v[2] : v[3]);
  };
  int epi_group = -1;
  Epi epi = kRows ? epi_in : epi_prepare(epi_in);

  // step -> panel, first token
  auto where = [&](int t, int& panel, long& q0) {
    const int s = s0 + t;
    if constexpr (kRows) panel = __builtin_amdgcn_readfirstlane((int)(((float)s + 0.5f) * inv_tq));   // (exact: s < 2^21, which the host sees to)
    else panel = x < a.more ? fastdiv(s, a.d_tq1) : fastdiv(s, a.d_tq);
    q0 = (long)TT * (tile0 + (s - panel * tq));
  };

  // ---- token tile -> LDS stage: instruction (kt, wave) = rows 8 wave .. + 7 of k-tile kt, chunk c of row r at slot
  // c ^ tfb_kc_swz(r) (the k-contiguous layout of the tiled kernels: conflict-free 128-bit fragment reads)
  // (tiles of 32 tokens: rows 8 (wave & 3) .. + 7 of the even or the odd k-tiles)
  const int w8 = TT == 64 ? wave : wave & 3, kt0 = TT == 64 ? 0 : wave >> 2;
  constexpr int KTS = TT == 64 ? 1 : 2;
  const uint32_t qv = (uint32_t)((lane >> 3) * a.Q.ld + (((lane & 7) ^ tfb_kc_swz((lane >> 3) + 8 * w8)) << 4));
  auto dma = [&](int t) {
    int panel;
    long q0;
    where(NS > 2 && t >= T ? T - 1 : t, panel, q0);   // (past the last tile that one again, into a stage nobody reads any more)
    const uint8_t* g = a.Q.base + (q0 + 8 * w8) * a.Q.ld + kt0 * 128;
    uint8_t* d = ring + (t & (NS - 1)) * STAGE + w8 * 1024 + kt0 * (TT * 128);
#pragma unroll
    for (int kt = 0; kt < NK; kt += KTS)
      __builtin_amdgcn_global_load_lds((tfb_glb_void_t*)(g + kt * 128 + (size_t)qv), (tfb_lds_void_t*)(d + kt * (TT * 128)), 16, 0, 0);
  };

  // ---- the panel's rows in registers: lane (lr, lh) holds bytes 64 ks + 32 lh .. + 31 of row 32 wave + lr per k-step
  // (loaded and waited for in inline assembly: behind compiler-visible loads the first MFMA of EVERY tile would wait for
  // all vector-memory operations in flight, the next tile's among them, because a run may have crossed a panel border)
  i32x4 Alo[KS], Ahi[KS];
  int cur_panel = -1, cur_group = 0;
  auto load_panel = [&](int panel, int group) __attribute__((always_inline)) {
    const uint8_t* g = a.P.base + (kRows ? group * a.p_group_stride : 0) + ((long)panel * 256 + 32 * wave + lr) * a.P.ld + 32 * lh;
#pragma unroll
    for (int ks = 0; ks < KS; ++ks) {
      asm volatile("global_load_dwordx4 %0, %1, off" : "=v"(Alo[ks]) : "v"(g + 64 * ks));
      asm volatile("global_load_dwordx4 %0, %1, off offset:16" : "=v"(Ahi[ks]) : "v"(g + 64 * ks));
    }
#pragma unroll
    for (int ks = 0; ks < KS; ks += 4)
      asm volatile("s_waitcnt vmcnt(0)"
                   : "+v"(Alo[ks]), "+v"(Ahi[ks]), "+v"(Alo[ks + 1]), "+v"(Ahi[ks + 1]), "+v"(Alo[ks + 2]), "+v"(Ahi[ks + 2]),
                     "+v"(Alo[ks + 3]), "+v"(Ahi[ks + 3]));
    cur_panel = panel;
    cur_group = group;
  };

  // ---- B fragment addresses in stage 0: token row lr (+ 32 j as an immediate), k-step 2 kt + u: chunks 4 u + 2 lh + e
  uint32_t ab[4];
  {
    const uint32_t lbase = (uint32_t)(size_t)(tfb_lds_u8*)ring;
    const int f = tfb_kc_swz(lr);
#pragma unroll
    for (int ue = 0; ue < 4; ++ue) {
      const int c = 4 * (ue >> 1) + 2 * lh + (ue & 1);
      ab[ue] = lbase + lr * 128 + (((c ^ f) & 7) << 4);
    }
  }

  uint8_t* stg = stg_all + (wave >> 1) * (TT * 256);

  // An epilogue's own operand (the saved activation of the dH GEMM) is requested when the wavefront starts to multiply the
  // tile and used one phase later: asked for in the epilogue itself, its round trip to HBM was that phase's length.
  constexpr bool kPrefetch = has_prefetch<Epi>::value;
  typedef typename prefetch_type<Epi>::type pre_t;
  [[maybe_unused]] pre_t pre[NP];

  // ---- one tile: KS NA MFMAs, the accumulators to the pair's staging block (row q = 256 bytes of fp32, 16-byte chunk c at
  // slot c ^ (q & 15))
  auto multiply = [&](int t) __attribute__((always_inline)) {
    int panel;
    long q0;
    where(t, panel, q0);
    if constexpr (kPrefetch) {
      const int p = panel * 256 + 64 * (wave >> 1) + 8 * (lane & 7), ql = (TT / 2) * (wave & 1) + (lane >> 3);
#pragma unroll
      for (int k = 0; k < NP; ++k) pre[k] = epi.prefetch(p, (int)q0 + ql + 8 * k);
    }
    if constexpr (NS > 2) dma(t + NS - 1);
    // (a tile that nobody has is multiplied with the weights at hand, and not finished)
    const int group = kRows ? group_at(q0) : 0;
    if ((panel != cur_panel || group != cur_group) && group >= 0) load_panel(panel, group);
    const uint32_t so = (t & (NS - 1)) * STAGE;
    f32x16 acc[NA];
#pragma unroll
    for (int j = 0; j < NA; ++j)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[j][e] = 0.f;
    // the fragments are read a k-step ahead of its MFMAs
    i32x4 b[2][2 * NA];
    auto rd = [&](auto KI) __attribute__((always_inline)) {
      constexpr int ks = decltype(KI)::value, off = (ks >> 1) * (TT * 128), u = ks & 1;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        b[u][e] = tfb_lds_read128<off, i32x4>(ab[2 * u + e] + so);
        if constexpr (NA == 2) b[u][2 + e] = tfb_lds_read128<off + 4096, i32x4>(ab[2 * u + e] + so);
      }
    };
    auto mm = [&](auto KI) __attribute__((always_inline)) {
      constexpr int ks = decltype(KI)::value;
      ws8_landed<NA, (ks + 1 < KS ? 2 * NA : 0)>(b[ks & 1]);
      const i32x4 al = Alo[ks], ah = Ahi[ks];
      const i32x8 av = {al.x, al.y, al.z, al.w, ah.x, ah.y, ah.z, ah.w};
#pragma unroll
      for (int j = 0; j < NA; ++j) {
        const i32x4 &lo = b[ks & 1][2 * j], &hi = b[ks & 1][2 * j + 1];
        const i32x8 bv = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
        acc[j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(av, bv, acc[j], FMTP, FMTQ, 0, 127, 0, 127);
      }
    };
    __builtin_amdgcn_s_setprio(1);
    rd(std::integral_constant<int, 0>{});
    ws8_unroll<0, KS>([&](auto KI) __attribute__((always_inline)) {
      constexpr int ks = decltype(KI)::value;
      if constexpr (ks + 1 < KS) rd(std::integral_constant<int, ks + 1>{});
      mm(KI);
    });
    __builtin_amdgcn_s_setprio(0);
    // acc[j][4 jj + e] = D[p = 8 jj + 4 lh + e][q = 32 j + lr]
    const int cw = 8 * (wave & 1) + lh;
#pragma unroll
    for (int jj = 0; jj < 4; ++jj)
#pragma unroll
      for (int j = 0; j < NA; ++j) {
        const f32x4 v = {acc[j][4 * jj], acc[j][4 * jj + 1], acc[j][4 * jj + 2], acc[j][4 * jj + 3]};
        *(f32x4*)(stg + (32 * j + lr) * 256 + (((cw + 2 * jj) ^ (lr & 15)) << 4)) = v;
      }
  };

  // ---- the epilogue of a tile: this wavefront's half of the pair's tokens, passes of 8 tokens x 64 p
  auto finish = [&](int t) __attribute__((always_inline)) {
    int panel;
    long q0;
    where(t, panel, q0);
    if constexpr (kRows) {
      const int group = group_at(q0);
      if (group < 0) return;
      if (group != epi_group) {
        epi = epi_prepare(epi_in.for_group(group));
        epi_group = group;
      }
    }
    const int p = panel * 256 + 64 * (wave >> 1) + 8 * (lane & 7);
    const int ql = (TT / 2) * (wave & 1) + (lane >> 3);
    [[maybe_unused]] long off = 0, down = 0;
    if constexpr (has_place<Epi>::value) {
      off = epi.place(p, (int)q0 + ql);
      down = epi.place(0, 8);
    }
#pragma unroll
    for (int k = 0; k < NP; ++k) {
      const int row = ql + 8 * k, c = 2 * (lane & 7);
      const f32x4 lo = *(const f32x4*)(stg + row * 256 + ((c ^ (row & 15)) << 4));
      const f32x4 hi = *(const f32x4*)(stg + row * 256 + (((c + 1) ^ (row & 15)) << 4));
      const float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
      if constexpr (has_place<Epi>::value) {
        if constexpr (kPrefetch) epi.put(off, v, pre[k]);
        else epi.put(off, v);
        off += down;
      } else if constexpr (kPrefetch) {
        epi(p, (int)q0 + row, v, pre[k], 0);
      } else {
        epi(p, (int)q0 + row, v, 0);
      }
    }
  };

  // ---- prologue: tile 0 on its way, the first panel into registers
#pragma unroll
  for (int t = 0; t < NS - 1; ++t) dma(t);
  {
    int panel;
    long q0;
    where(0, panel, q0);
    load_panel(panel, kRows ? max(group_at(q0), 0) : 0);
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  TFB_SBAR();

  // Phase ph: group 0 multiplies tile ph / 2 (ph even) or finishes it (ph odd); group 1 one phase later. Tile t + 1 is
  // requested in phase 2 t - by group 0 in front of its MFMAs, by group 1 behind its epilogue - into the stage whose tile
  // (t - 1) group 1 stopped reading in phase 2 t - 1, and waited for in phase 2 t + 1, a phase after the request: by group 1
  // behind its MFMAs with nothing younger outstanding, by group 0 in front of its epilogue, where only the epilogue's own
  // four operand loads (if it has any) are younger - behind the epilogue the wait would be for its stores' round trips
  // (completion is reported in issue order, stores included).
  // Four stages: tile t + 3 is requested by a group when it multiplies tile t, behind the epilogue's operand loads (so that these can be
  // waited for without it), and tile t + 1 waited for at the same places, where the loads of the two tiles after it are younger.
  for (int ph = 0; ph <= 2 * T; ++ph) {
    if ((ph & 1) == grp) {
      const int t = (ph - grp) >> 1;
      if (t < T) {
        if (NS == 2 && grp == 0 && t + 1 < T) dma(t + 1);
        multiply(t);
        if (grp == 1) {
          if (NS > 2) asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * ND) : "memory");
          else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        }
      }
    } else {
      const int t = (ph - 1 - grp) >> 1;  // group 0: (ph - 1) / 2; group 1: (ph - 2) / 2
      if (NS > 2 && grp == 0) {
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"((NS - 2) * ND) : "memory");
      } else if (grp == 0) {
        if (kPrefetch) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NP) : "memory");
        else asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      }
      if (ph - 1 - grp >= 0 && t < T) finish(t);
      if (NS == 2 && grp == 1) {
        const int tn = (ph >> 1) + 1;
        if (tn < T) dma(tn);
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the staging block is complete (or read) before the roles swap
    TFB_SBAR();
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// np % 256 == 0, nq % 128 == 0, kbytes == 768 or 1024, rows 16-byte aligned; at least eight steps of 64 tokens for every CU: a
// workgroup loads its weight panel and fills its pipeline once per run, and a shorter run does not pay for that against the tiled
// kernels (up-projection / dH, us, this kernel against them: 768 x 3072, 2048 tokens 14.5 / 18.0 against 10.6 / 13.9, 8192 tokens 32.4 /
// 42.6 against 29.5 / 40.0, 12288 tokens 41.6 / 52.9 against 43.9 / 57.2; 1024 x 4096, 8192 tokens 50 / 56 against 57 / 69, 9600 tokens 59 /
// 67 against 69 / 83, 16384 tokens 87 / 99 against 113 / 127; 1024 x 2816, 32768 tokens 118 / 132 against 130 / 154).
static inline bool gemm_ws8_applies(long np, long nq, long kbytes) {
  return TFB_WS8 && (kbytes == 768 || kbytes == 1024) && np > 0 && nq > 0 && np % 256 == 0 && nq % 128 == 0 &&
         (np / 256) * (nq / 64) >= 8L * tfb_resident_slots(1);
}

// ... over the rows of groups: twice as many steps, for a run also loads the weights of each of its groups (us, this kernel against the tiled one,
// up-projection / dH of eight experts with the same load, then with two that have nearly all: 1024 x 2816, 12288 rows 60 / 66 against 69 / 69 and
// 72 / 77 against 65 / 75; 24576 rows 111 / 119 against 132 / 134 and 122 / 126 against 122 / 128; 768 x 3072, 11264 rows 47 / 55 against
// 46 / 59 and 52 / 61 against 46 / 59; 32768 rows 103 / 119 against 155 / 152 and 120 / 121 against 156 / 155; 1024 x 4096, 32768 rows 173 / 180
// against 274 / 273; sixteen experts, 1024 x 2816, 32768 rows 138 / 149 against 167 / 172).
static inline bool gemm_ws8_rows_applies(long np, long nq, long kbytes) {
  return gemm_ws8_applies(np, nq, kbytes) && nq <= WS8_ROWS_MAX && (np / 256) * (nq / 64) >= 16L * tfb_resident_slots(1) &&
         (np / 256) * (nq / 32) < (1L << 21);
}

// K1024: also contractions of 1024 bytes.
template <int FMTP, int FMTQ, bool K1024, class Epi>
static int gemm_ws8_launch(GemmOperand P, GemmOperand Q, int np, int nq, long kbytes, Epi epi, hipStream_t stream,
                           const int* row_group = nullptr, long p_group_stride = 0) {
  if (has_rows<Epi>::value && (!row_group || !gemm_ws8_rows_applies(np, nq, kbytes) || (p_group_stride & 15))) return TFB_ERR_SHAPE;
  if ((kbytes != 768 && (!K1024 || kbytes != 1024)) || np <= 0 || nq <= 0 || np % 256 || nq % 128) return TFB_ERR_SHAPE;
  if (P.ld <= 0 || Q.ld <= 0 || P.ld > (1L << 24) || Q.ld > (1L << 24)) return TFB_ERR_SHAPE;
  if (((uintptr_t)P.base | (uintptr_t)Q.base | (uintptr_t)P.ld | (uintptr_t)Q.ld) & 15) return TFB_ERR_ARG;
  Ws8Args a = {};
  a.P = P;
  a.Q = Q;
  a.row_group = row_group;
  a.p_group_stride = p_group_stride;
  a.row_tiles = nq / 128;
  const int tiles = nq / (kbytes == 768 ? 64 : 32);
  a.panels = np / 256;
  a.tq = tiles / 8;
  a.more = tiles % 8;
  if ((long)a.panels * (a.tq + 1) >= (1L << 30)) return TFB_ERR_SHAPE;
  const int steps_x = a.panels * (a.tq + (a.more ? 1 : 0));
  int per_x = tfb_resident_slots(1) / 8;  // workgroups per XCD: one per CU
  if (per_x < 1) per_x = 1;
  a.per_wg = (steps_x + per_x - 1) / per_x;
  const int wgs_x = has_rows<Epi>::value ? per_x : (steps_x + a.per_wg - 1) / a.per_wg;
  a.d_tq = fastdiv_make(a.tq > 0 ? a.tq : 1);
  a.d_tq1 = fastdiv_make(a.tq + 1);
  auto go = [&](auto nk) {
    hipLaunchKernelGGL((gemm_ws8_kernel<decltype(nk)::value, FMTP, FMTQ, Epi>), dim3(8 * wgs_x), dim3(512), 0, stream, a, epi);
    TFB_LAUNCH_CHECK();
    return (int)TFB_OK;
  };
  if constexpr (K1024)
    if (kbytes == 1024) return go(std::integral_constant<int, 8>{});
  return go(std::integral_constant<int, 6>{});
}
