// Persistent 256 x 256 MFMA GEMM for gfx950: D[p][q] = sum_k P[p][k] * Q[q][k], fp32 accumulation, k-contiguous operands.
//
// One workgroup of eight wavefronts per CU (two per SIMD) walks output tiles. The wavefronts form two groups of four (one
// wavefront of each group on every SIMD) that alternate between a MEMORY cluster (fragment reads from LDS, operand loads
// global -> LDS) and an MFMA cluster (8 MFMAs of 32 x 32), one barrier per cluster, group 1 running one cluster behind
// group 0: each SIMD's matrix pipe is fed by one wavefront while the other one waits on the memory path, and a vector
// memory instruction (which holds the wavefront that issues it for 70-110 cycles) never delays an MFMA.
//
// A wavefront owns 2 x 64 rows of P (64 in each 128-row half of the tile) and 2 x 32 rows of Q: four accumulator blocks of
// 64 x 32. A k-tile (128 bytes of k per row) is consumed as: block (P half 0, Q half 0), (0, 1), (1, 0), (1, 1); an operand
// quarter (128 rows x 128 bytes = 16 KB, one of P half 0/1, Q half 0/1) is refilled with the k-tile two ahead as soon as
// both groups have it in registers, so two 64 KB stages keep the loads ~1.5 k-tiles ahead of the MFMAs. The load stream
// does not stop at an output tile's end: the last two k-tiles of a tile already fetch the first two of the workgroup's next
// tile, and the epilogue (accumulators -> bf16 -> global, straight from registers: a lane pair exchange with
// v_permlane32_swap gives every lane 8 consecutive outputs of a row) runs while those loads are in flight.
//
// Narrow tiles (192 x 256, 256 x 192) fill rounds of the CUs that 256 x 256 leaves part empty: an output of 768 columns is four tiles
// of 192, so 16384 rows are 256 tiles instead of 192. The operand with 192 rows is the one of which a wavefront owns two halves; of the
// second it then owns one MFMA tile, and the two blocks of that half share a cluster: six clusters a k-tile, every one 8 MFMAs.
//
// Fragment reads are inline assembly (ds_read_b128 with immediate offsets) with explicit s_waitcnt: left to the compiler,
// every LDS read beside global -> LDS loads in flight would wait for vmcnt(0).
//
// LDS map (bytes): stage S at S * 65536: P half 0, P half 1, Q half 0, Q half 1 (16 KB each). A k-contiguous operand
// ([rows][K]) keeps row r of a half at r * 128, 16-byte chunk c at slot c ^ tfb_kc_swz(r) (no bank conflicts for the 128-bit
// fragment reads). A k-strided bf16 operand ([K][rows], the token-contraction GEMMs) keeps one k per 256-byte LDS row,
// chunk c of k-row k at slot c ^ (4 (k & 3)), and its fragments come through ds_read_b64_tr_b16 (two per fragment), the
// layout and lane map of the 128 x 128 kernel's K_STRIDED reader. A k-strided fp8 operand keeps one k per 128-byte LDS row
// (128 k-rows per quarter), chunk c of k-row k at slot c ^ (2 ((k >> 1) & 3)), fragments through ds_read_b64_tr_b8 (four
// per 64-k fragment).
//
// Long contractions with few output tiles (the LM head's gradients: 384 tiles of 512 k-tiles) are split along k into
// work items of equal length; each leaves its fp32 partial tile in a workspace (epilogues with kSplitF32, staged as
// fp32) and splitk_reduce_kernel finishes them.
#pragma once
#include "gemm_core.hpp"

typedef __attribute__((address_space(3))) uint8_t tfb_lds_u8;
typedef unsigned tfb_u32x2 __attribute__((ext_vector_type(2)));

template <int OFF, class T>
__device__ __forceinline__ T tfb_lds_read128(uint32_t addr) {
  static_assert(sizeof(T) == 16, "128-bit fragment");
  T v;
  asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
  return v;
}
#define TFB_SBAR()                          \
  do {                                      \
    __builtin_amdgcn_sched_barrier(0);      \
    asm volatile("s_barrier" ::: "memory"); \
    __builtin_amdgcn_sched_barrier(0);      \
  } while (0)

struct PpArgs {
  GemmOperand P, Q;
  int nk_total; // k-tiles of the contraction; split s of `splits` takes [s nk / splits, (s + 1) nk / splits), >= 2 each
  int ntiles;   // work items = output tiles * splits (item w: split w / nout, output tile w % nout)
  int nout;     // output tiles
  int splits;
  int ipx;      // > 0 (k ranges of one round; slow tile rows that are no multiple of 8): XCD x (= workgroup & 7) takes the ipx consecutive
                // work items from x * ipx, so that an XCD's workgroups share k ranges or slow rows of the operands in its L2
  FastDiv d_nout;
  int nwg;      // workgroups launched (a multiple of 8 when rect)
  int p_fast;   // the fast-walking operand is P
  int nfast;    // tiles of that operand
  // rect: XCD x (= work item & 7) owns R consecutive tile rows of the slow operand and walks them in panels of GW
  // columns (GW * R ~ the XCD's 32 CUs), so the tiles that run together on an XCD form a compact block and share their
  // operand rows in that XCD's L2
  int rect, R, GW, panel;  // panel = GW * R
  int gw_last;             // width of the last panel (nfast % GW, or GW)
  FastDiv d_nfast, d_panel, d_gw, d_gw_last;
  // Two contractions of the same rows (an epilogue with kExperts): output tiles from nout0 on are the second's
  GemmOperand P1, Q1;
  int nout0, p_fast1, nfast1;
  FastDiv d_nfast1;
  // over segments of them: group e's is seg[e] .. seg[e + 1], multiples of 128 rows. A workgroup has one output tile of one group:
  // XCD x tiles x ipx .. of the group with the most rows, then of the next
  const int* seg;
  int ngroups;
  FastDiv d_ipx;
  // over row tiles of groups (an epilogue with kRows): row_group[t] names the group of rows 128 t .. (-1: nobody's), its P lies
  // p_group_stride bytes further
  const int* row_group;
  int row_tiles;
  long p_group_stride;
};
template <class T, class = void>
struct has_experts : std::false_type {};
template <class T>
struct has_experts<T, std::void_t<decltype(T::kExperts)>> : std::true_type {};

template <class T, class = void>
struct has_rows : std::false_type {};
template <class T>
struct has_rows<T, std::void_t<decltype(T::kRows)>> : std::true_type {};

// A value that no store of this launch changes, by a scalar load (a vector load would be waited for behind the operand loads in flight)
template <class T>
__device__ __forceinline__ T tfb_scalar_load(const T* p) {
  return *(const __attribute__((address_space(4))) T*)(uintptr_t)p;
}

// The grouped rows of a launch with kRows, cut into items of 256 rows from every group's first (128 where its last tile is alone), and what
// the persistent kernel takes of the output tiles (256 columns of an item; item by item): whole rounds of the `nwg` workgroups, and a last part
// of one too when it is 0.3 of a round or more (or the only one); what it leaves is finished by the ring (gemm_ring_rest_kernel). Only
// the device knows the groups' loads; every wavefront reads the table for itself (64 tiles a lane-chunk, up to 4096 tiles).
struct RowItems {
  unsigned long long starts;  // lane c: the tiles among 64 c .. 64 c + 63 at which an item starts
  int before;                 // lane c: the items that start in front of those
  int items, total, taken;    // items; output tiles; those of the persistent kernel
  bool ragged;                // it leaves some
  __device__ __forceinline__ void init(const int* group, int tiles, int ncol, int nwg, int lane) {
    starts = 0;
    before = items = 0;
    int seg0 = 0;  // the first tile of the group that a chunk begins in
    for (int c0 = 0; 64 * c0 < tiles; c0 += 4) {
      int g[4], gp[4];
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int i = 64 * (c0 + x) + lane;
        g[x] = i < tiles ? group[i] : -1;
        gp[x] = i > 0 && i < tiles ? group[i - 1] : -1;
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        const int c = c0 + x, i = 64 * c + lane;
        const unsigned long long b = __ballot(i == 0 || g[x] != gp[x]), le = b & (~0ull >> (63 - lane));
        const int s0 = le ? 64 * c + 63 - __builtin_clzll(le) : seg0;
        const unsigned long long m = __ballot(g[x] >= 0 && ((i - s0) & 1) == 0);
        if (lane == c) {
          starts = m;
          before = items;
        }
        items += __builtin_popcountll(m);
        if (b) seg0 = 64 * c + 63 - __builtin_clzll(b);
      }
    }
    total = items * ncol;
    const int full = total / nwg, rest = total - full * nwg;
    ragged = full > 0 && rest > 0 && 10 * rest < 3 * nwg;
    taken = ragged ? full * nwg : total;
    chunks = (tiles + 63) >> 6;
  }
  int chunks;
  // the first tile of item k
  __device__ __forceinline__ int tile(int k, int lane) const {
    const int c = 63 - __builtin_clzll(__ballot(lane < chunks && before <= k));
    const unsigned lo = __builtin_amdgcn_readlane((unsigned)starts, c), hi = __builtin_amdgcn_readlane((unsigned)(starts >> 32), c);
    const int r = k - __builtin_amdgcn_readlane(before, c), below = __builtin_amdgcn_mbcnt_hi(hi, __builtin_amdgcn_mbcnt_lo(lo, 0));
    const unsigned bit = lane < 32 ? lo >> lane : hi >> (lane - 32);
    return 64 * c + __builtin_ctzll(__ballot((bit & 1) && below == r));
  }
};

// Epilogue protocol of this kernel (every epilogue of the library rounds f(accumulator) to bf16 first):
//   float pre(float acc)                      applied to every accumulator before its rounding to bf16;
//   void chunk(p, q, v [, pre_t])             8 consecutive rounded outputs D[p .. p + 7][q] as four packed bf16 pairs (p % 8 == 0);
//                                             with a pre_t (16 bytes) the operand from at(p, q) that the chunk needs;
//   void chunk2(p, q, lo, hi, a, b)           with kPartner: the outputs from p and those kPartner (32 or 64) further on, a and b
//                                             the 16 bytes from at(p, q) and at2(p, q).
typedef short tfb_s16x8 __attribute__((ext_vector_type(8)));
template <int OFF>
__device__ __forceinline__ tfb_s16x4 tfb_lds_read_tr64(uint32_t addr) {
  tfb_s16x4 v;
  asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
  return v;
}
typedef int tfb_pp_i32x2 __attribute__((ext_vector_type(2)));
template <int OFF>
__device__ __forceinline__ tfb_pp_i32x2 tfb_lds_read_tr64_b8(uint32_t addr) {
  tfb_pp_i32x2 v;
  asm volatile("ds_read_b64_tr_b8 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
  return v;
}

// An epilogue with the static member kSplitF32 receives the raw fp32 accumulators, operator()(p, q, v[8], split): the
// partial tile of a k-split.
template <class T, class = void>
struct has_split_f32 : std::false_type {};
template <class T>
struct has_split_f32<T, std::void_t<decltype(T::kSplitF32)>> : std::true_type {};

// SHAPE: the output tile, rows of p x rows of q.
#define TFB_PP_256x256 0
#define TFB_PP_192x256 1
#define TFB_PP_256x192 2

// ES: element size (2: bf16, 1: OCP fp8 with FMTP / FMTQ = 0 e4m3, 1 e5m2 per side); LAYP / LAYQ: TFB_K_CONTIG or
// TFB_K_STRIDED
template <int ES, int FMTP, int FMTQ, int LAYP, int LAYQ, class Epi, int SHAPE = TFB_PP_256x256>
__global__ __launch_bounds__(512, 2) void gemm_pp_kernel(PpArgs a, Epi epi_in) {
  constexpr bool kF32 = has_split_f32<Epi>::value;
  // X is the operand of which a wavefront owns up to 2 x 64 rows (wr), Y the one of which it owns 2 x 32 (wc)
  constexpr bool NARROW = SHAPE != TFB_PP_256x256, QX = SHAPE == TFB_PP_256x192;
  constexpr int TP = SHAPE == TFB_PP_192x256 ? 192 : 256, TQ = QX ? 192 : 256;
  constexpr int LAYX = QX ? LAYQ : LAYP, LAYY = QX ? LAYP : LAYQ;
  constexpr int kPartner = partner_of<Epi>::value;
  static_assert(!NARROW || (!kF32 && !has_experts<Epi>::value && !kPartner), "a narrow tile's half 1 has 32 rows of a wavefront");
  // A partner 64 outputs away: a wavefront's two MFMA tiles of a P half are rows 32 wr .. and 64 + 32 wr ..
  constexpr int XROWS = kPartner == 64 ? 32 : 64, XTILE = kPartner == 64 ? 64 : 32;  // rows of X from one group to the other; from tile i = 0 to 1
  static_assert(kPartner != 64 || LAYX == TFB_K_CONTIG, "the fragments' rows");
  constexpr bool kRows = has_rows<Epi>::value;
  static_assert(!kRows || (!NARROW && !kF32 && LAYP == TFB_K_CONTIG && LAYQ == TFB_K_CONTIG && !has_prefetch<Epi>::value), "rows of groups");
  constexpr bool kPipe = has_prefetch<Epi>::value;  // the epilogue reads an operand of its own
  static_assert(!NARROW || LAYX == TFB_K_CONTIG || ES == 2, "half a quarter of fp8 rows");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[2 * 65536];
  __shared__ __attribute__((aligned(1024))) uint8_t stg_all[8 * 4096];  // epilogue staging, 4 KB per wavefront
  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), lane = tid & 63;
  const int wr = wave >> 2, wc = wave & 3;  // wr: the group (wavefronts 0-3 / 4-7 sit on SIMDs 0-3 each)
  const int lr = lane & 31, lh = lane >> 5;
  int nkt;  // k-tiles of the current work item
  uint8_t* stg = stg_all + wave * 4096;

  // ---- operand loads. A quarter is 16 instructions of 1 KB, two per wavefront (g = wave and wave + 8):
  //   k-contiguous: instruction g = rows 8 g .. 8 g + 7 x 128 bytes of k, lane l -> row l / 8, chunk (l % 8) ^ swizzle;
  //   k-strided:    instruction g = k-rows 4 g .. 4 g + 3 x 128 rows (256 bytes), lane l -> k-row l / 16, chunk (l % 16) ^ 4 (k & 3);
  //                 fp8: k-rows 8 g .. 8 g + 7 x 128 rows (128 bytes), lane l -> k-row l / 8, chunk (l % 8) ^ 2 ((k >> 1) & 3).
  // Per operand: v = the lane's byte offset, istep = from instruction g to g + 8, hstep = from half 0 to half 1,
  // kstep = from one k-tile to the next, and the byte origin of output tile row-block r0.
  struct Side {
    const uint8_t* base;  // operand base + this wavefront's first instruction
    uint32_t v;
    long istep, hstep, kstep, tstep;  // tstep: bytes per row of the output tile origin
  };
  auto make_side = [&](const GemmOperand& o, int lay) {
    Side sd;
    if (lay == TFB_K_CONTIG) {
      const int lrow = lane >> 3;
      const int dch = (lane & 7) ^ tfb_kc_swz(lrow + 8 * wave);
      sd.base = o.base + 8L * wave * o.ld;
      sd.v = (uint32_t)(lrow * o.ld + dch * 16);
      sd.istep = 64 * o.ld;
      sd.hstep = 128 * o.ld;
      sd.kstep = 128;
      sd.tstep = o.ld;
    } else if (ES == 2) {
      const int kl = lane >> 4, slot = lane & 15;
      sd.base = o.base + 4L * wave * o.ld;
      sd.v = (uint32_t)(kl * o.ld + ((slot ^ (4 * kl)) << 4));
      sd.istep = 32 * o.ld;
      sd.hstep = 256;
      sd.kstep = 64 * o.ld;
      sd.tstep = 2;
    } else {
      const int kl = lane >> 3, slot = lane & 7;
      sd.base = o.base + 8L * wave * o.ld;
      sd.v = (uint32_t)(kl * o.ld + ((slot ^ (2 * ((kl >> 1) & 3))) << 4));
      sd.istep = 64 * o.ld;
      sd.hstep = 128;
      sd.kstep = 128 * o.ld;
      sd.tstep = 1;
    }
    return sd;
  };
  [[maybe_unused]] int first = 0;  // the first output tile of this workgroup's contraction
  [[maybe_unused]] int group_tile = 0, group_k0 = 0, group_nkt = 0;
  if constexpr (has_experts<Epi>::value) {
    const int j = blockIdx.x >> 3, rank = fastdiv(j, a.d_ipx);
    group_tile = (blockIdx.x & 7) * a.ipx + j - rank * a.ipx;
    if (group_tile >= a.nout) return;  // (whole workgroup)
    // the group of that rank: more rows first, of equal ones the lower index
    const int rows = lane < a.ngroups ? a.seg[lane + 1] - a.seg[lane] : -1;
    int before = 0;
    for (int m = 0; m < a.ngroups; ++m) {
      const int other = __builtin_amdgcn_readlane(rows, m);
      before += other > rows || (other == rows && m < lane);
    }
    const int group = __builtin_ctzll(__ballot(lane < a.ngroups && before == rank));
    group_k0 = __builtin_amdgcn_readfirstlane(a.seg[group]) / 128;
    group_nkt = __builtin_amdgcn_readlane(rows, group) / 128;
    epi_in = epi_in.for_group(group);
    if (group_tile >= a.nout0) {
      first = a.nout0;
      a.P = a.P1;
      a.Q = a.Q1;
      a.p_fast = a.p_fast1;
      a.nfast = a.nfast1;
      a.d_nfast = a.d_nfast1;
      epi_in = epi_in.for_second();
    }
  }
  const Side sx = make_side(QX ? a.Q : a.P, LAYX), sy = make_side(QX ? a.P : a.Q, LAYY);
  [[maybe_unused]] RowItems ri;
  if constexpr (kRows) ri.init(a.row_group, a.row_tiles, a.nfast, a.nwg, lane);
  [[maybe_unused]] int row_group = 0;      // kRows, of the item that tile_of was last asked for: its group,
  [[maybe_unused]] bool row_alone = false; // and whether its second 128 rows are not its group's

  // work item -> output tile origin and split
  auto tile_of = [&](int w, long& p0, long& q0, int& split) {
    split = 0;
    if (a.splits > 1) {
      split = fastdiv(w, a.d_nout);
      w -= split * a.nout;
    }
    if constexpr (has_experts<Epi>::value) w -= first;
    if constexpr (kRows) {
      const int k = fastdiv(w, a.d_nfast), t = __builtin_amdgcn_readfirstlane(ri.tile(k, lane));
      row_group = tfb_scalar_load(a.row_group + t);
      row_alone = t + 1 >= a.row_tiles || tfb_scalar_load(a.row_group + t + 1) != row_group;
      p0 = (long)(w - k * a.nfast) * TP;
      q0 = (long)t * 128;
      return;
    }
    int fast, slow;
    if (a.rect) {
      const int x = w & 7, j = w >> 3;
      const int pn = fastdiv(j, a.d_panel), rem = j - pn * a.panel;
      const int first = pn * a.GW;
      const bool last = first + a.GW > a.nfast;
      const int row = last ? fastdiv(rem, a.d_gw_last) : fastdiv(rem, a.d_gw);
      const int gw = last ? a.gw_last : a.GW;
      fast = first + rem - row * gw;
      slow = x * a.R + row;
    } else {
      slow = fastdiv(w, a.d_nfast);
      fast = w - slow * a.nfast;
    }
    p0 = (long)(a.p_fast ? fast : slow) * TP;
    q0 = (long)(a.p_fast ? slow : fast) * TQ;
  };
  auto krange = [&](int split, int& k0, int& n) {
    k0 = 0;
    n = a.nk_total;
    if constexpr (has_experts<Epi>::value) {
      k0 = group_k0;
      n = group_nkt;
    }
    if (a.splits > 1) {
      k0 = (int)((long)split * a.nk_total / a.splits);
      n = (int)((long)(split + 1) * a.nk_total / a.splits) - k0;
    }
  };
  auto origin = [&](const Side& sd, long r0, int k0) { return sd.base + r0 * sd.tstep + (long)k0 * sd.kstep; };

  // quarter (X / Y, half h) of stage S <- the k-tile at g (the side's address of that k-tile of the output tile). The 64 rows of a
  // narrow tile's X half 1: k-contiguous, the first instruction alone; k-strided, both with the lanes of the chunks beyond them off.
  [[maybe_unused]] const bool in_half = ((lane & 15) ^ (4 * (lane >> 4))) < 8;
  // (alone, kRows: rows 128 .. 255 of the Y tile are another group's or no one's; the first 128 come twice, and are not stored again)
  auto dma = [&](int S, int Y, int h, const uint8_t* g, bool alone = false) __attribute__((always_inline)) {
    const Side& sd = Y ? sy : sx;
    uint8_t* d = lds + S * 65536 + Y * 32768 + h * 16384 + wave * 1024;
    const bool half = NARROW && !Y && h;
    if (half && LAYX == TFB_K_STRIDED && !in_half) return;
#pragma unroll
    for (int i = 0; i < (half && LAYX == TFB_K_CONTIG ? 1 : 2); ++i)
      __builtin_amdgcn_global_load_lds((tfb_glb_void_t*)(g + (kRows && alone ? 0 : h * sd.hstep) + i * sd.istep + (size_t)sd.v),
                                       (tfb_lds_void_t*)(d + i * 8192), 16, 0, 0);
  };
  constexpr int NX1 = NARROW && LAYX == TFB_K_CONTIG ? 1 : 2;  // a wavefront's load instructions for X half 1

  // ---- fragment addresses (stage 0; the stage bit is toggled after every k-tile)
  uint32_t ax[4], ay[4];
  [[maybe_unused]] uint32_t ax1[4];  // of X half 1 of a narrow tile, where a wavefront's rows are wr * 32 ..
  {
    const uint32_t lbase = (uint32_t)(size_t)(tfb_lds_u8*)lds;
    const int rx = wr * XROWS + lr, rx1 = wr * 32 + lr, ry = wc * 32 + lr;
    // k-contiguous, one address per k-step. bf16: k-step s (16 k) of a row is chunk 2 s + lh; fp8: k-step s (64 k) is
    // chunks 4 s + 2 lh, + 1: entry 2 s + u
#pragma unroll
    for (int s = 0; s < 4; ++s) {
      const int c = ES == 2 ? 2 * s + lh : 4 * (s >> 1) + 2 * lh + (s & 1);
      ax[s] = lbase + rx * 128 + (((c ^ tfb_kc_swz(rx)) & 7) << 4);
      ax1[s] = lbase + rx1 * 128 + (((c ^ tfb_kc_swz(rx1)) & 7) << 4);
      ay[s] = lbase + 32768 + ry * 128 + (((c ^ tfb_kc_swz(ry)) & 7) << 4);
    }
    // k-strided: 16-lane group g4 reads rows 16 (g4 & 1) .. + 15 of an MFMA tile, k-group g4 >> 1; lane j of the group
    // points at k-row j / 4 (of four consecutive k), rows 4 (j % 4) .. + 3. One address per 32-row tile (ax[0], ax[1]:
    // the second tile's chunk index differs in bit 2, which the swizzle also touches, so it is not an immediate offset);
    // k-step s is 16 k-rows further (an immediate), the fragment's upper four k another 4 k-rows.
    const int g4 = lane >> 4, j = lane & 15, kq = j >> 2;
    // fp8: lane j of the group points at k-row j / 2 (of eight consecutive k), rows 8 (j % 2) .. + 7; the group's k-half
    // is 32 k-rows further, a k-step 64, the fragment's next eight k 8 (immediates).
    auto tr_addr = [&](int row0) {
      if (ES == 2) {
        const int p = row0 + 16 * (g4 & 1) + 4 * (j & 3);
        return (uint32_t)((8 * (g4 >> 1) + kq) * 256 + ((((p >> 3) ^ (4 * kq)) << 4) | ((p & 4) << 1)));
      }
      const int p = row0 + 16 * (g4 & 1) + 8 * (j & 1), k8 = j >> 1;
      return (uint32_t)((32 * (g4 >> 1) + k8) * 128 + ((((p >> 4) ^ (2 * ((k8 >> 1) & 3))) << 4) | (p & 8)));
    };
    if (LAYX == TFB_K_STRIDED) {
      ax[0] = lbase + tr_addr(wr * 64);
      ax[1] = lbase + tr_addr(wr * 64 + 32);
      ax1[0] = lbase + tr_addr(wr * 32);
    }
    if (LAYY == TFB_K_STRIDED) ay[0] = lbase + 32768 + tr_addr(wc * 32);
  }
  // addresses in use
  constexpr int NAX = LAYX == TFB_K_STRIDED ? 2 : 4, NAX1 = !NARROW ? 0 : LAYX == TFB_K_STRIDED ? 1 : 4, NAY = LAYY == TFB_K_STRIDED ? 1 : 4;

  f32x16 acc[2][2][2];  // [X half][i][Y half]
  // fragments: bf16 four k-steps of 16 (one 128-bit read each), fp8 two k-steps of 64 (two 128-bit reads each)
  typedef std::conditional_t<ES == 2, bf16x8, i32x4> r128_t;
  r128_t fa[2][4], fb0[4], fb1[4];
  auto tr_frag = [&](auto OFF, uint32_t addr) {
    constexpr int off = decltype(OFF)::value;
    if constexpr (ES == 2) {  // k-step off / 4096: 16 k-rows of 256 bytes; the upper four k 4 rows further
      const tfb_s16x4 lo = tfb_lds_read_tr64<off>(addr), hi = tfb_lds_read_tr64<off + 1024>(addr);
      const tfb_s16x8 v = {lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
      return __builtin_bit_cast(r128_t, v);
    } else {  // half a 64-k fragment: 16 k of a row, two reads 8 k-rows (1 KB) apart
      const tfb_pp_i32x2 lo = tfb_lds_read_tr64_b8<off>(addr), hi = tfb_lds_read_tr64_b8<off + 1024>(addr);
      return r128_t{lo.x, lo.y, hi.x, hi.y};
    }
  };
  // fragment entry e (bf16: k-step e of 16 k; fp8: half e & 1 of k-step e >> 1 of 64 k) -> byte offset in a quarter
  constexpr int TR1 = ES == 2 ? 4096 : 2048, TR2 = 8192, TR3 = ES == 2 ? 12288 : 8192 + 2048;
  auto readA = [&](auto H) __attribute__((always_inline)) {
    constexpr int h = decltype(H)::value;
    if constexpr (NARROW && h) {
      if constexpr (LAYX == TFB_K_CONTIG) {
#pragma unroll
        for (int s = 0; s < 4; ++s) fa[0][s] = tfb_lds_read128<16384, r128_t>(ax1[s]);
      } else {
        fa[0][0] = tr_frag(std::integral_constant<int, 16384>{}, ax1[0]);
        fa[0][1] = tr_frag(std::integral_constant<int, 16384 + TR1>{}, ax1[0]);
        fa[0][2] = tr_frag(std::integral_constant<int, 16384 + TR2>{}, ax1[0]);
        fa[0][3] = tr_frag(std::integral_constant<int, 16384 + TR3>{}, ax1[0]);
      }
    } else if constexpr (LAYX == TFB_K_CONTIG) {
#pragma unroll
      for (int s = 0; s < 4; ++s) {
        fa[0][s] = tfb_lds_read128<h * 16384, r128_t>(ax[s]);
        fa[1][s] = tfb_lds_read128<h * 16384 + XTILE * 128, r128_t>(ax[s]);
      }
    } else {
      fa[0][0] = tr_frag(std::integral_constant<int, h * 16384>{}, ax[0]);
      fa[1][0] = tr_frag(std::integral_constant<int, h * 16384>{}, ax[1]);
      fa[0][1] = tr_frag(std::integral_constant<int, h * 16384 + TR1>{}, ax[0]);
      fa[1][1] = tr_frag(std::integral_constant<int, h * 16384 + TR1>{}, ax[1]);
      fa[0][2] = tr_frag(std::integral_constant<int, h * 16384 + TR2>{}, ax[0]);
      fa[1][2] = tr_frag(std::integral_constant<int, h * 16384 + TR2>{}, ax[1]);
      fa[0][3] = tr_frag(std::integral_constant<int, h * 16384 + TR3>{}, ax[0]);
      fa[1][3] = tr_frag(std::integral_constant<int, h * 16384 + TR3>{}, ax[1]);
    }
  };
  // flip = 0x10000: the fragments of the OTHER stage (the next k-tile)
  auto readB = [&](auto H, r128_t(&fb)[4], uint32_t flip = 0) __attribute__((always_inline)) {
    constexpr int h = decltype(H)::value;
    if constexpr (LAYY == TFB_K_CONTIG) {
#pragma unroll
      for (int s = 0; s < 4; ++s) fb[s] = tfb_lds_read128<h * 16384, r128_t>(ay[s] ^ flip);
    } else {
      fb[0] = tr_frag(std::integral_constant<int, h * 16384>{}, ay[0] ^ flip);
      fb[1] = tr_frag(std::integral_constant<int, h * 16384 + TR1>{}, ay[0] ^ flip);
      fb[2] = tr_frag(std::integral_constant<int, h * 16384 + TR2>{}, ay[0] ^ flip);
      fb[3] = tr_frag(std::integral_constant<int, h * 16384 + TR3>{}, ay[0] ^ flip);
    }
  };
  // the fragments pass through the wait as in/out operands, so that no MFMA that reads them is scheduled ahead of it
  auto waitA = [&]() {
    asm volatile("s_waitcnt lgkmcnt(0)"
                 : "+v"(fa[0][0]), "+v"(fa[0][1]), "+v"(fa[0][2]), "+v"(fa[0][3]), "+v"(fa[1][0]), "+v"(fa[1][1]),
                   "+v"(fa[1][2]), "+v"(fa[1][3]));
  };
  auto waitA1 = [&]() {  // (X half 1 of a narrow tile: one tile of 32 rows)
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(fa[0][0]), "+v"(fa[0][1]), "+v"(fa[0][2]), "+v"(fa[0][3]));
  };
  auto waitB = [&](r128_t(&fb)[4]) {
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(fb[0]), "+v"(fb[1]), "+v"(fb[2]), "+v"(fb[3]));
  };
  auto mma = [&](auto FIRST, auto HX, auto HY, const r128_t(&fb)[4]) __attribute__((always_inline)) {
    constexpr bool first = decltype(FIRST)::value;
    constexpr int hx = decltype(HX)::value, hy = decltype(HY)::value, NI = NARROW && hx ? 1 : 2;
    __builtin_amdgcn_s_setprio(1);
#pragma unroll
    for (int s = 0; s < (ES == 2 ? 4 : 2); ++s)
#pragma unroll
      for (int i = 0; i < NI; ++i) {
        f32x16 c = acc[hx][i][hy];
        if (first && s == 0) {
#pragma unroll
          for (int e = 0; e < 16; ++e) c[e] = 0.f;
        }
        // the P fragment is the MFMA's A operand
        if constexpr (ES == 2) {
          acc[hx][i][hy] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(QX ? fb[s] : fa[i][s], QX ? fa[i][s] : fb[s], c, 0, 0, 0);
        } else {
          const i32x4 xl = fa[i][2 * s], xh = fa[i][2 * s + 1], yl = fb[2 * s], yh = fb[2 * s + 1];
          const i32x8 xv = {xl.x, xl.y, xl.z, xl.w, xh.x, xh.y, xh.z, xh.w};
          const i32x8 yv = {yl.x, yl.y, yl.z, yl.w, yh.x, yh.y, yh.z, yh.w};
          // formats: 0 = e4m3, 1 = e5m2; E8M0 scale byte 127 = 2^0
          acc[hx][i][hy] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(QX ? yv : xv, QX ? xv : yv, c, FMTP, FMTQ, 0, 127, 0, 127);
        }
      }
    __builtin_amdgcn_s_setprio(0);
    // the MFMAs have no side effects: without a use here they may sink below the barriers that follow
    if constexpr (NI == 2) asm volatile("" : "+v"(acc[hx][0][hy]), "+v"(acc[hx][1][hy]));
    else asm volatile("" : "+v"(acc[hx][0][hy]));
  };
  typedef std::integral_constant<int, 0> H0;
  typedef std::integral_constant<int, 1> H1;

  Epi epi = epi_prepare(epi_in);
  int w = blockIdx.x, w_step = a.nwg, w_end = a.ntiles;  // this workgroup's items: w, w + w_step, .. below w_end
  if constexpr (has_experts<Epi>::value) {
    w = group_tile;
    w_end = 0;
  } else if constexpr (kRows) {  // consecutive tiles for an XCD
    const int per = (ri.taken + 7) >> 3, x0 = (w & 7) * per;
    w = x0 + (w >> 3);
    w_step = a.nwg >> 3;
    w_end = x0 + per < ri.taken ? x0 + per : ri.taken;
    if (w >= w_end) return;  // (whole workgroup)
  } else if (a.ipx > 0) {
    const int x0 = (w & 7) * a.ipx;
    w = x0 + (w >> 3);
    w_step = a.nwg >> 3;
    w_end = x0 + a.ipx < a.ntiles ? x0 + a.ipx : a.ntiles;
    if (w >= w_end) return;  // (whole workgroup)
  }
  long p0, q0;
  int split, k0;
  tile_of(w, p0, q0, split);
  krange(split, k0, nkt);
  const uint8_t* gx = origin(sx, QX ? q0 : p0, k0);  // current work item: the sides' addresses of its first k-tile
  const uint8_t* gy = origin(sy, QX ? p0 : q0, k0);
  [[maybe_unused]] bool alone = row_alone, alone_next = false, alone_prev = false;
  [[maybe_unused]] Epi epi_now = epi, epi_next = epi;  // kRows: of this item and the next (epi: of the one that is stored)
  if constexpr (kRows) {
    gx += row_group * a.p_group_stride;
    epi_now = epi_prepare(epi_in.for_group(row_group));
  }

  // A segment without rows: nothing is loaded, its product is zero.
  if constexpr (has_experts<Epi>::value) {
    if (nkt == 0) {
      const float v[8] = {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f};
      for (int i = tid; i < 256 * 32; i += 512) epi((int)p0 + 8 * (i & 31), (int)q0 + (i >> 5), v, 0);
      return;
    }
  }

  // ---- prologue: all of k-tile 0 into stage 0, three quarters of k-tile 1 into stage 1 (narrow tiles: the two quarters 0)
  dma(0, 1, 0, gy);
  dma(0, 0, 0, gx);
  dma(0, 1, 1, gy, alone);
  dma(0, 0, 1, gx);
  const long k_one = has_experts<Epi>::value && nkt < 2 ? 0 : 1;  // (a segment of one k-tile: that one again)
  dma(1, 0, 0, gx + k_one * sx.kstep);
  dma(1, 1, 0, gy + k_one * sy.kstep);
  if constexpr (!NARROW) dma(1, 1, 1, gy + k_one * sy.kstep, alone);
  asm volatile("s_waitcnt vmcnt(%0)" ::"n"(NARROW ? 4 : 6) : "memory");
  TFB_SBAR();               // k-tile 0 is there for everybody
  if (wr == 1) TFB_SBAR();  // group 1 runs one cluster behind from here on

  // ---- epilogue of one accumulator block, acc[hx][i][hy][4 jj + e] = D[pb + 8 jj + 4 lh + e][qb + lr] of MFMA tile i: every
  // accumulator goes through epi.pre() and is rounded to bf16, the block passes through the wavefront's own 4 KB of LDS, and every
  // lane finishes 8 consecutive outputs of a row (with kPartner those and their partners): epi.chunk() or epi.chunk2(). Two forms:
  //   64 p (X = P, two tiles): row q = 128 bytes, 16-byte chunk c at slot c ^ ((q >> 1) & 7) (the 8-byte writes and the 16-byte
  //   reads then use the banks evenly), a row's 64 outputs on 8 consecutive lanes;
  //   32 p: row q = 64 bytes, chunk c at slot c ^ ((q >> 2) & 3), a row's outputs on 4 lanes; X = Q: tile i is rows 32 i .. of q.
  // The epilogue's own operand (a residual, rotation tables) is four 16-byte loads a lane and block, requested one store ahead by request_pre().
  u32x4 pre[8] = {};  // (the second four only behind the loop)
  auto here = [](int x) __attribute__((always_inline)) {  // (what is made of it is not kept in registers across the loop)
    if constexpr (kPipe) asm volatile("" : "+v"(x));
    return x;
  };
  auto load_pre = [&](int k, const void* g) __attribute__((always_inline)) {
    if constexpr (kPartner) asm volatile("global_load_dwordx4 %0, %1, off" : "+v"(pre[k]) : "v"(g) : "memory");
    else asm volatile("global_load_dwordx4 %0, %1, off nt" : "+v"(pre[k]) : "v"(g) : "memory");  // (read once)
  };
  auto wait_pre = [&](auto AFTER, auto FROM) __attribute__((always_inline)) {  // AFTER: vector memory instructions issued since
    auto* r = pre + decltype(FROM)::value;
    asm volatile("s_waitcnt vmcnt(%4)" : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]) : "n"(decltype(AFTER)::value) : "memory");
  };
  // a block's place: its first p and q, a lane's chunk and first row, rows from one of its chunks to the next, chunks
  auto block_p = [&](auto HX, auto HY, long tp0) { return (int)tp0 + (QX ? decltype(HY)::value * 128 + wc * 32
                                                                         : decltype(HX)::value * 128 + wr * (NARROW && decltype(HX)::value ? 32 : XROWS)); };
  auto block_q = [&](auto HX, auto HY, long tq0) { return (int)tq0 + (QX ? decltype(HX)::value * 128 + wr * (NARROW && decltype(HX)::value ? 32 : 64)
                                                                         : decltype(HY)::value * 128 + wc * 32); };
  auto request_pre = [&](auto HX, auto HY, long tp0, long tq0, auto FROM) __attribute__((always_inline)) {
    constexpr int hx = decltype(HX)::value, NI = NARROW && hx ? 1 : 2, from = decltype(FROM)::value;
    constexpr bool wide = !QX && NI == 2 && !kPartner;
    constexpr int NCH = wide ? 4 : kPartner ? 2 : QX ? 2 * NI : 2, RSTEP = wide ? 8 : 16;
    const int ln = here(lane), p = block_p(HX, HY, tp0) + 8 * (wide ? ln & 7 : ln & 3), q = block_q(HX, HY, tq0) + (wide ? ln >> 3 : ln >> 2);
    if constexpr (kPipe) {
#pragma unroll
      for (int k = 0; k < NCH; ++k) {
        if constexpr (kPartner != 0) {
          load_pre(from + 2 * k, epi.at(p, q + RSTEP * k));
          load_pre(from + 2 * k + 1, epi.at2(p, q + RSTEP * k));
        } else {
          load_pre(from + k, epi.at(p, q + RSTEP * k));
        }
      }
    }
  };
  auto store_block = [&](auto HX, auto HY, long tp0, long tq0, auto FROM) __attribute__((always_inline)) {
    constexpr int hx = decltype(HX)::value, hy = decltype(HY)::value, NI = NARROW && hx ? 1 : 2, from = decltype(FROM)::value;
    constexpr bool wide = !QX && NI == 2;
    const int pb = block_p(HX, HY, tp0), qb = block_q(HX, HY, tq0), ln = here(lane);
#pragma unroll
    for (int i = 0; i < NI; ++i)
#pragma unroll
      for (int jj = 0; jj < 4; ++jj) {
        const f32x16& c = acc[hx][i][hy];
        if constexpr (!kF32) {
          u32x2 v = {pack2bf(epi.pre(c[4 * jj + 0]), epi.pre(c[4 * jj + 1])),
                     pack2bf(epi.pre(c[4 * jj + 2]), epi.pre(c[4 * jj + 3]))};
          if constexpr (wide) *(u32x2*)(stg + lr * 128 + (((4 * i + jj) ^ ((lr >> 1) & 7)) << 4) + 8 * lh) = v;
          else *(u32x2*)(stg + (32 * i + lr) * 64 + ((jj ^ ((lr >> 2) & 3)) << 4) + 8 * lh) = v;
        }
      }
    __builtin_amdgcn_wave_barrier();
    if constexpr (kPartner != 0) {  // a lane takes a chunk of the block's first 32 outputs and its partner together
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int row = (ln >> 2) + 16 * k, ch = ln & 3;
        const u32x4 lo = *(const u32x4*)(stg + row * 128 + ((ch ^ ((row >> 1) & 7)) << 4));
        const u32x4 hi = *(const u32x4*)(stg + row * 128 + (((ch + 4) ^ ((row >> 1) & 7)) << 4));
        if constexpr (!kF32) epi.chunk2(pb + 8 * ch, qb + row, lo, hi, pre[from + 2 * k], pre[from + 2 * k + 1]);
      }
    } else {
      constexpr int NCH = wide ? 4 : QX ? 2 * NI : 2, RSTEP = wide ? 8 : 16;  // chunks of a lane, rows apart
      const int ch = wide ? ln & 7 : ln & 3, row0 = wide ? ln >> 3 : ln >> 2;
#pragma unroll
      for (int k = 0; k < NCH; ++k) {
        const int row = row0 + RSTEP * k;
        const u32x4 v = wide ? *(const u32x4*)(stg + row * 128 + ((ch ^ ((row >> 1) & 7)) << 4))
                             : *(const u32x4*)(stg + row * 64 + ((ch ^ ((row >> 2) & 3)) << 4));
        if constexpr (kPipe) epi.chunk(pb + 8 * ch, qb + row, v, pre[from + k]);
        else if constexpr (!kF32) epi.chunk(pb + 8 * ch, qb + row, v);
      }
    }
    __builtin_amdgcn_wave_barrier();
  };

  // The same for the partial tile of a k-split (epilogues with kSplitF32): sixteen output rows at a time pass through the
  // 4 KB as fp32 (row = 256 bytes, 16-byte chunk c at slot c ^ row), and a lane finishes 8 consecutive fp32 outputs.
  auto store_block_f32 = [&](auto HP, auto HQ, long tp0, long tq0, int sp_) __attribute__((always_inline)) {
    constexpr int hp = decltype(HP)::value, hq = decltype(HQ)::value;
    const int pb = (int)tp0 + hp * 128 + wr * 64, qb = (int)tq0 + hq * 128 + wc * 32;
    const int ch = lane & 7, r8 = lane >> 3;
#pragma unroll
    for (int qh = 0; qh < 2; ++qh) {
      if ((lr >> 4) == qh) {
        const int row = lr & 15;
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int jj = 0; jj < 4; ++jj) {
            const f32x16& c = acc[hp][i][hq];
            const f32x4 v = {c[4 * jj + 0], c[4 * jj + 1], c[4 * jj + 2], c[4 * jj + 3]};
            *(f32x4*)(stg + row * 256 + (((8 * i + 2 * jj + lh) ^ row) << 4)) = v;
          }
      }
      __builtin_amdgcn_wave_barrier();
#pragma unroll
      for (int k = 0; k < 2; ++k) {
        const int row = r8 + 8 * k;
        const f32x4 lo = *(const f32x4*)(stg + row * 256 + (((2 * ch) ^ row) << 4));
        const f32x4 hi = *(const f32x4*)(stg + row * 256 + (((2 * ch + 1) ^ row) << 4));
        const float v[8] = {lo[0], lo[1], lo[2], lo[3], hi[0], hi[1], hi[2], hi[3]};
        if constexpr (kF32) epi(pb + 8 * ch, qb + 16 * qh + row, v, sp_);
      }
      __builtin_amdgcn_wave_barrier();
    }
  };

  int S = 0;
  readB(H0{}, fb0);
  bool have_prev = false;  // the previous tile's accumulators are still to be stored
  long pp0 = 0, pq0 = 0;   // its origin
  // the workgroup's next work item (its first k-tiles are requested by this one's last iterations); past the end: this
  // one again (loads nobody reads, from valid memory)
  int wn, splitn, k0n, nktn;
  long pn, qn;
  const uint8_t *gxn, *gyn;
  auto look_ahead = [&]() __attribute__((always_inline)) {
    wn = w + w_step;
    pn = p0;
    qn = q0;
    splitn = split;
    k0n = k0;
    nktn = nkt;
    if (wn < w_end) {
      tile_of(wn, pn, qn, splitn);
      krange(splitn, k0n, nktn);
    }
    gxn = origin(sx, QX ? qn : pn, k0n);
    gyn = origin(sy, QX ? pn : qn, k0n);
    if constexpr (kRows) {
      alone_next = row_alone;
      gxn += row_group * a.p_group_stride;
      epi_next = epi_prepare(epi_in.for_group(row_group));
    }
  };
  auto go_on = [&]() __attribute__((always_inline)) {
    p0 = pn;
    q0 = qn;
    split = splitn;
    k0 = k0n;
    nkt = nktn;
    gx = gxn;
    gy = gyn;
    if constexpr (kRows) {
      alone = alone_next;
      epi_now = epi_next;
    }
  };
  // One k-tile. In a tile's first iteration the MFMAs start from zero, and each accumulator block of the PREVIOUS tile is
  // stored in the memory cluster in front of the MFMA cluster that overwrites it: the stores of one group (4 KB per
  // wavefront and cluster) run under the other group's MFMAs. An epilogue with an operand of its own (kPipe) has it requested behind the
  // stores of the cluster before (the first block's in the tile's last iteration) and in front of that cluster's operand loads: reported in issue
  // order, it does not wait for them. Requested in its own cluster behind those loads, every one of a tile's four blocks waited for a trip to
  // HBM (the QKV projection with its rotation, 32768 x 2304 x 768: 148 us, of 113 without; now 120). The requests take the registers as
  // operands that go in and come out, which leaves no reason for a copy of them while a load is on its way; that none is made, and none of the
  // registers used, is checked in the built code (tests/test_built_code_waits.py).
  auto iter = [&](auto FIRST, int kt) __attribute__((always_inline)) {
    constexpr bool first = decltype(FIRST)::value, stores = first && !kF32;
    // k positions one and two ahead in the workgroup's stream of k-tiles
    const bool in1 = kt + 1 < nkt, in2 = kt + 2 < nkt;
    const long k1 = in1 ? kt + 1 : 0, k2 = in2 ? kt + 2 : has_experts<Epi>::value && nkt < 2 ? 0 : kt + 2 - nkt;
    const uint8_t* gx1 = (in1 ? gx : gxn) + k1 * sx.kstep;
    const uint8_t* gx2 = (in2 ? gx : gxn) + k2 * sx.kstep;
    const uint8_t* gy2 = (in2 ? gy : gyn) + k2 * sy.kstep;
    auto store = [&](auto HX, auto HY, auto FROM) __attribute__((always_inline)) {
      if constexpr (stores) {
        if (have_prev && !(kRows && decltype(HY)::value == 1 && alone_prev)) store_block(HX, HY, pp0, pq0, FROM);
      }
    };
    // kPipe: the block whose operand was requested before AFTER vector memory instructions; then next() asks for the next one's
    auto store_pipe = [&](auto HX, auto HY, auto AFTER, auto next) __attribute__((always_inline)) {
      if constexpr (stores && kPipe) {
        if (have_prev) {
          wait_pre(AFTER, H0{});
          store_block(HX, HY, pp0, pq0, H0{});
          next();
        }
      }
    };
    auto store_plain = [&](auto HX, auto HY) __attribute__((always_inline)) {
      if constexpr (!kPipe) store(HX, HY, H0{});
    };
    auto request_first = [&]() __attribute__((always_inline)) {
      if constexpr (kPipe && !first) {
        if (!in1) request_pre(H0{}, H0{}, p0, q0, H0{});
      }
    };
    auto nothing = []() {};
    typedef std::integral_constant<int, 2> N2;
    if constexpr (!NARROW) {
      // c0 (the Y fragments of half 0 were requested in the previous k-tile's c7)
      readA(H0{});
      store_pipe(H0{}, H0{}, N2{}, [&]() { request_pre(H0{}, H1{}, pp0, pq0, H0{}); });
      dma(S ^ 1, 0, 1, gx1);
      store_plain(H0{}, H0{});
      TFB_SBAR();
      // c1
      waitB(fb0);
      waitA();
      mma(FIRST, H0{}, H0{}, fb0);
      TFB_SBAR();
      // c2
      readB(H1{}, fb1);
      store_pipe(H0{}, H1{}, N2{}, [&]() { request_pre(H1{}, H0{}, pp0, pq0, H0{}); });
      dma(S, 0, 0, gx2);
      store_plain(H0{}, H1{});
      TFB_SBAR();
      // c3
      waitB(fb1);
      mma(FIRST, H0{}, H1{}, fb1);
      TFB_SBAR();
      // c4
      readA(H1{});
      store_pipe(H1{}, H0{}, N2{}, [&]() { request_pre(H1{}, H1{}, pp0, pq0, H0{}); });
      dma(S, 1, 0, gy2);
      store_plain(H1{}, H0{});
      TFB_SBAR();
      // c5
      waitA();
      mma(FIRST, H1{}, H0{}, fb0);
      // Completion is reported in issue order, stores included. Everything up to the quarter requested in c0 has to be
      // there one cluster before the other group's matching wait: all but the two quarters requested since (4
      // instructions), and in a first iteration with stores all but those and the 12 stores (c0's four were issued
      // behind its loads); kPipe: c2's and c4's stores and four requests each, in front of their loads. After the barrier that ends c6 both
      // groups have waited, so the next k-tile is complete.
      if (kRows && stores && have_prev && alone_prev) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");  // (c2 has stored nothing)
      else if (stores && have_prev) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(kPipe ? 20 : 16) : "memory");
      else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      TFB_SBAR();
      // c6
      store_pipe(H1{}, H1{}, N2{}, nothing);
      request_first();
      dma(S, 1, 1, gy2, in2 ? alone : alone_next);
      store_plain(H1{}, H1{});
      TFB_SBAR();
      // c7: the next k-tile's first Y fragments are requested under this cluster's MFMAs (fb0 was last read in c5)
      readB(H0{}, fb0, 0x10000u);
      mma(FIRST, H1{}, H1{}, fb1);
      TFB_SBAR();
    } else {
      // X half 1 is one MFMA tile a wavefront: three MFMA clusters of 8 instead of four. Quarters 0 are requested two k-tiles
      // ahead, quarters 1 one ahead. A cluster's reads are waited for in front of its barrier (the requests behind them take longer),
      // so a quarter is requested again only when a barrier has passed since either group had the old one in registers.
      const uint8_t* gy1 = (in1 ? gy : gyn) + k1 * sy.kstep;
      // c0 (Y half 0: see c5)
      readA(H0{});
      store_pipe(H0{}, H0{}, std::integral_constant<int, 4>{}, [&]() { request_pre(H0{}, H1{}, pp0, pq0, H0{}); });
      dma(S ^ 1, 1, 1, gy1);
      dma(S ^ 1, 0, 1, gx1);
      store_plain(H0{}, H0{});
      waitB(fb0);
      waitA();
      TFB_SBAR();
      // c1
      mma(FIRST, H0{}, H0{}, fb0);
      TFB_SBAR();
      // c2
      readB(H1{}, fb1);
      store_pipe(H0{}, H1{}, std::integral_constant<int, 2 + NX1>{}, [&]() {
        request_pre(H1{}, H0{}, pp0, pq0, H0{});
        request_pre(H1{}, H1{}, pp0, pq0, N2{});
      });
      store_plain(H0{}, H1{});
      waitB(fb1);
      TFB_SBAR();
      // c3
      mma(FIRST, H0{}, H1{}, fb1);
      // The next k-tile's quarters 0 (requested in the previous iteration's c4) have to be there: all but what was requested
      // since, c0's loads and in a first iteration with stores the 8 stores of c0 and c2, kPipe: and their eight requests. c5 reads them
      // behind two more barriers.
      if (stores && have_prev) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 + NX1 + (kPipe ? 16 : 8)) : "memory");
      else asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 + NX1) : "memory");
      TFB_SBAR();
      // c4
      readA(H1{});
      store_pipe(H1{}, H0{}, H0{}, [&]() { store_block(H1{}, H1{}, pp0, pq0, N2{}); });
      request_first();
      dma(S, 0, 0, gx2);
      dma(S, 1, 0, gy2);
      store_plain(H1{}, H0{});
      store_plain(H1{}, H1{});
      waitA1();
      TFB_SBAR();
      // c5
      mma(FIRST, H1{}, H0{}, fb0);
      readB(H0{}, fb0, 0x10000u);
      mma(FIRST, H1{}, H1{}, fb1);
      // The next k-tile's quarters 1 (c0) likewise: all but c4's four loads, and with stores the 8 of c0 and c2 and c4's 4. (kPipe: c4 has
      // waited for them.)
      if (stores && have_prev) asm volatile("s_waitcnt vmcnt(16)" ::: "memory");
      else asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      TFB_SBAR();
    }
    S ^= 1;
#pragma unroll
    for (int s = 0; s < NAX; ++s) ax[s] ^= 0x10000u;
#pragma unroll
    for (int s = 0; s < NAX1; ++s) ax1[s] ^= 0x10000u;
#pragma unroll
    for (int s = 0; s < NAY; ++s) ay[s] ^= 0x10000u;
  };
  for (;;) {
    look_ahead();
    iter(std::true_type{}, 0);
    if constexpr (has_experts<Epi>::value) {
      for (int kt = 1; kt < nkt; ++kt) iter(std::false_type{}, kt);
    } else {
      int kt = 1;
      do iter(std::false_type{}, kt);
      while (++kt < nkt);
    }
    if constexpr (kF32) {
      // a k-split's partial tile: stored here, both groups together (a work item is hundreds of k-tiles long)
      if (wr == 0) TFB_SBAR();  // group 0 waits for group 1's last cluster
      store_block_f32(H0{}, H0{}, p0, q0, split);
      store_block_f32(H0{}, H1{}, p0, q0, split);
      store_block_f32(H1{}, H0{}, p0, q0, split);
      store_block_f32(H1{}, H1{}, p0, q0, split);
    } else {
      have_prev = true;
      pp0 = p0;
      pq0 = q0;
      if constexpr (kRows) {
        alone_prev = alone;
        epi = epi_now;
      }
    }
    w = wn;
    if (w >= w_end) break;
    go_on();
    if constexpr (kF32) {
      if (wr == 1) TFB_SBAR();  // group 1 falls one cluster behind again
    }
  }
  if constexpr (!kF32) {
    waitB(fb0);  // the stream's last fragments, which nobody multiplies, land before their registers are used again
    // the last tile's accumulators
    if constexpr (kPipe) {
      // Each block's operand is requested in front of the stores of the block before it, into the other four registers. Behind them its wait
      // covered those stores as well, three times a launch (us, bf16 with a residual: 12288 x 1024 x 1024 37.6 -> 35.3, 10240 x 1024 x 1024 36.2 -> 33.8,
      // 4096 x 3072 x 1024 37.0 -> 34.6; fp8 20480 x 512 x 2048 32.9 -> 30.2, 12288 x 768 x 3072 35.5 -> 33.1; 10240 x 1536 with its rotation 24.8 -> 23.7).
      constexpr int HALF = NARROW ? 2 : 4;  // requests and stores of a block of half 1; half 0: four
      typedef std::integral_constant<int, 4> N4;
      request_pre(H0{}, H1{}, pp0, pq0, N4{});
      wait_pre(N4{}, H0{});
      store_block(H0{}, H0{}, pp0, pq0, H0{});
      request_pre(H1{}, H0{}, pp0, pq0, H0{});
      wait_pre(std::integral_constant<int, 4 + HALF>{}, N4{});
      store_block(H0{}, H1{}, pp0, pq0, N4{});
      request_pre(H1{}, H1{}, pp0, pq0, N4{});
      wait_pre(std::integral_constant<int, 4 + HALF>{}, H0{});
      store_block(H1{}, H0{}, pp0, pq0, H0{});
      wait_pre(std::integral_constant<int, HALF>{}, N4{});
      store_block(H1{}, H1{}, pp0, pq0, N4{});
    } else {
      store_block(H0{}, H0{}, pp0, pq0, H0{});
      if (!(kRows && alone_prev)) store_block(H0{}, H1{}, pp0, pq0, H0{});
      store_block(H1{}, H0{}, pp0, pq0, H0{});
      if (!(kRows && alone_prev)) store_block(H1{}, H1{}, pp0, pq0, H0{});
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // the stream's last (unused) loads must have landed before LDS is released
}

// Shapes this kernel takes: np, nq multiples of 256 (192 on a narrow tile's side), at least two k-tiles of 128 bytes.
// Shapes it is USED for: its tiles have to fill their rounds of the CUs, to 60 % where there is one round and to 70 % otherwise,
// because a CU works on one tile at a time; then the half operand traffic per output wins against the 128 x 128 kernel at every
// contraction length (standalone, us, that kernel -> this one): bf16 2048 x 32768 x 768 (4.0 rounds) 140 -> 105, 8192 x 4096 x 768
// (2.0) 69 -> 51, 10240 x 1024 x 768 (0.62) 27.8 -> 23.8, 16384 x 768 x 2304 (0.75) 78 -> 58; fp8 16384 x 3072 x 1024 (3.0) 69 -> 50;
// at the line 8192 x 3072 x 768 (1.5) 46.4 -> 47.2, and below it 8192 x 2304 x 768 (1.12) 37.6 -> 41.8, 8192 x 1024 x 768 (0.5)
// 18.5 -> 23.7. A heavy epilogue per tile (residual add, the MLP's activation) is serial with the k-loop here and runs
// under another workgroup's MFMAs there: those need 16 k-tiles or 4096 tiles as well (in the training step, 6 to 12 k-tiles:
// 55 -> 60, 112 -> 111 us); 24 on a narrow tile (bf16 32768 x 768 x 768 with a residual 49.9 -> 51.4, 16384 rows 27.2 -> 28.3).
// The rotary embedding's tables are the same few for all heads, asked for ahead and out of the L2: it goes by the plain rule with lines 1.04 as
// high (K 768, N 2304: 6144 rows 31.7 -> 28.3, 12288 56.1 -> 49.7, 16384 70.4 -> 68.2, 20480 90 -> 76, 32768 149 -> 120; N 1536, K 512: 10240
// 24.6 -> 22.6, 32768 70.8 -> 58.7; N 768, K 256: 16384 17.6 -> 16.7, 65536 51.7 -> 38.3; at the plain lines 10240 x 2304 46.1 -> 47.5).
// A narrow tile takes 0.75 / 0.92 (192 x 256) or 0.75 / 0.84 (256 x 192) of a 256 x 256 tile's time, so it is taken where its rounds save
// that much (us, the kernel of before -> this one): fp8 16384 x 768 x 3072 40.9 -> 36.8, 32768 rows 73.0 -> 65.5, 9600 x 1024 x 4096 51.7 ->
// 40.3, 11904 x 768 x 3072 50.6 -> 30.3; bf16 32768 x 768 x 2304 118 -> 104, 30336 x 768 x 768 55 -> 43, 12672 x 768 x 3072 95 -> 62; not in
// place of a 256 x 256 launch of as many rounds for 256 x 192 (fp8 11520 x 1024 x 2816 38.2 -> 40.3). Against the 128 x 128 kernel: its two
// workgroups a CU run a round in 0.65 of a 256 x 256 tile's time, half a round or less (one a CU) in 0.38 (4992 x 1536 x 1536, 0.91 of a
// round: 28.6 there, 34.9 here).
#ifndef TFB_PP
#define TFB_PP 1  // 0: every GEMM on the 128 x 128 kernel; 2: every shape the kernel takes (for comparisons)
#endif
#ifndef TFB_PP_SHAPE
#define TFB_PP_SHAPE -1  // 0, 1, 2: that tile only (for comparisons)
#endif
// The tile for an output of np x nq, or -1: the one that keeps the CUs busiest (256 x 256 also for all but the last 128 rows of q, where
// it has a full round without them: a launch of the ring more, 0.15 of a round).
// line: of the shares of their rounds that the tiles have to fill, for an epilogue between a plain and a heavy one.
static inline int gemm_pp_shape(long np, long nq, long kbytes, bool heavy_epilogue, bool narrow_ok, double line = 1.0) {
  if (!TFB_PP || np <= 0 || nq <= 0 || kbytes < 256 || kbytes % 128) return -1;
  const long cus = tfb_resident_slots(1);
  const double core_rounds = (double)((np + 127) / 128) * (double)((nq + 127) / 128) / (double)(2 * cus), whole = (double)(long)core_rounds;
  const double core = 0.65 * whole + (core_rounds == whole ? 0.0 : core_rounds - whole > 0.5 ? 0.65 : 0.38);
  int best = -1;
  double best_cost = 1e30, whole_tiles = 1e30;
  for (int shape = 0; shape < (narrow_ok ? 3 : 1); ++shape) {
    if (TFB_PP_SHAPE >= 0 && shape != TFB_PP_SHAPE) continue;
    const long tp = shape == TFB_PP_192x256 ? 192 : 256, tq = shape == TFB_PP_256x192 ? 192 : 256;
    const long rest = nq % tq, tiles = (np / tp) * (nq / tq), rounds = (tiles + cus - 1) / cus;
    if (np % tp || tiles < 8 || (rest && (shape || rest != 128 || tiles < cus))) continue;
    const double cost = (double)rounds * (shape == 0 ? 1.0 : shape == TFB_PP_192x256 ? 0.75 / 0.92 : 0.75 / 0.84) + (rest ? 0.15 : 0.0);
    if (TFB_PP != 2 && TFB_PP_SHAPE < 0) {
      if ((double)tiles < (rounds == 1 ? 0.6 : 0.7) * line * (double)(rounds * cus)) continue;
      if (heavy_epilogue && kbytes / 128 < (shape ? 24 : 16) && tiles < 4096) continue;
      if (shape && (cost > (heavy_epilogue ? 0.9 : 0.95) * core || cost > 0.88 * whole_tiles)) continue;
    }
    if (shape == 0) whole_tiles = cost;
    if (cost < best_cost) {
      best_cost = cost;
      best = shape;
    }
  }
  return best;
}

// np, nq multiples of the tile; kbytes = the contraction in bytes of a k-contiguous row (elements * ES), a multiple of 128
// with at least two k-tiles per split. With splits > 1 the epilogue is one with kSplitF32 (EpiSplit); when all work items
// fit one round of the CUs they are dealt to the XCDs in consecutive runs (PpArgs::ipx).
template <int ES, int FMTP, int FMTQ, int LAYP, int LAYQ, int SHAPE = TFB_PP_256x256, class Epi>
static int gemm_pp_launch_lay(GemmOperand P, GemmOperand Q, int np, int nq, long kbytes, int splits, Epi epi, hipStream_t stream) {
  constexpr int TP = SHAPE == TFB_PP_192x256 ? 192 : 256, TQ = SHAPE == TFB_PP_256x192 ? 192 : 256;
  if (np <= 0 || nq <= 0 || splits <= 0 || np % TP || nq % TQ || kbytes % 128 || kbytes / 128 / splits < 2)
    return TFB_ERR_SHAPE;
  if (P.ld <= 0 || Q.ld <= 0 || P.ld > (1L << 28) || Q.ld > (1L << 28)) return TFB_ERR_SHAPE;
  if (((uintptr_t)P.base | (uintptr_t)Q.base | (uintptr_t)P.ld | (uintptr_t)Q.ld) & 15) return TFB_ERR_ARG;
  if ((splits > 1) != has_split_f32<Epi>::value) return TFB_ERR_ARG;
  PpArgs a = {};
  a.P = P;
  a.Q = Q;
  a.splits = splits;
  a.nk_total = (int)(kbytes / 128);
  const int ntp = np / TP, ntq = nq / TQ;
  if ((long)ntp * ntq * splits >= (1L << 30)) return TFB_ERR_SHAPE;
  a.nout = ntp * ntq;
  a.ntiles = a.nout * splits;
  const int cus = tfb_resident_slots(1);
  a.p_fast = np <= nq;
  a.nfast = a.p_fast ? ntp : ntq;
  const int nslow = a.p_fast ? ntq : ntp;
  a.rect = (nslow % 8 == 0) && a.nout >= 8;
  a.nwg = a.ntiles < cus ? a.ntiles : cus;
  // Slow rows that are no multiple of 8: consecutive items per XCD too while it can keep the fast operand beside them (us, dealt over the
  // XCDs one by one -> so: fp8 16128 x 768 x 3072 on 192 x 256 tiles 45.8 -> 35; bf16 12032 x 2304 x 768 51.3 -> 47.5, 9600 x 3072 x 1024 65.6 ->
  // 64.7, 18816 x 4096 x 1024 156.3 -> 155.8; 9600 x 8192 x 1024, 16.8 MB, 154.6 -> 159.4).
  const long fast_bytes = (long)(a.p_fast ? np : nq) * kbytes;
  if (splits > 1 ? a.ntiles <= cus : !a.rect && a.ntiles >= 8 && fast_bytes <= (8L << 20) + (1L << 19)) {
    a.rect = 0;
    a.ipx = (a.ntiles + 7) / 8;
    a.nwg = 8 * a.ipx < cus ? 8 * a.ipx : cus & ~7;
  }
  if (a.rect) a.nwg &= ~7;
  if (a.nwg <= 0) return TFB_ERR_SHAPE;
  a.R = a.rect ? nslow / 8 : 1;
  // panel width: GW * R ~ the 32 workgroups an XCD runs together; a narrow fast operand (<= 4 tiles) is walked whole, so
  // that the tiles sharing a row block of the slow operand run together
  int gw = a.R >= 32 ? 1 : (32 + a.R - 1) / a.R;
  if (a.R > 8 && a.R < 32) gw = 32 / a.R > 0 ? 32 / a.R : 1;
  if (gw > a.nfast || a.nfast <= 4) gw = a.nfast;
  a.GW = gw;
  a.panel = a.GW * a.R;
  a.gw_last = a.nfast % a.GW ? a.nfast % a.GW : a.GW;
  a.d_nfast = fastdiv_make(a.nfast);
  a.d_panel = fastdiv_make(a.panel);
  a.d_gw = fastdiv_make(a.GW);
  a.d_gw_last = fastdiv_make(a.gw_last);
  a.d_nout = fastdiv_make(a.nout);
  hipLaunchKernelGGL((gemm_pp_kernel<ES, FMTP, FMTQ, LAYP, LAYQ, Epi, SHAPE>), dim3(a.nwg), dim3(512), 0, stream, a, epi);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}

// k ranges for a long contraction (nkt k-tiles) over fewer than 64 output tiles of 256 x 256, one work item per workgroup:
// up to 32 tiles, as many ranges per XCD as its CUs have room for tiles (an XCD's workgroups then read one k range of the
// operands together: 27 tiles -> 8 ranges, 9 tiles -> 24); beyond, the count that fills the CUs. 0: not worth it (less
// than 80 % of the CUs busy, fewer than 16 k-tiles per item, or the partial tiles do not fit the workspace).
static inline int gemm_pp_fewtile_splits(long t256, long nkt, long out_elems, long ws_bytes) {
  const long cus = tfb_resident_slots(1);
  if (t256 <= 0 || t256 >= 64) return 0;
  int c = t256 * 8 <= cus ? 8 * (int)(cus / 8 / t256) : (int)(cus / t256);
  while (c > 1 && (nkt / c < 16 || (long)c * out_elems * 4 > ws_bytes)) --c;
  return (c > 1 && (double)(t256 * c) >= 0.8 * (double)cus) ? c : 0;
}

// Two weight gradients of each of `groups` experts over its rows: P_i e4m3, Q_i e5m2, row segments seg (device, multiples of 128 rows). The
// experts' loads are the router's and often far apart: tiles of the heaviest expert first, so that the others' fill the CUs beside its long
// ones (and both gradients in one launch, so that these are twice as many).
template <class Epi>
static int gemm_pp_launch_experts(GemmOperand P0, GemmOperand Q0, int np0, int nq0, GemmOperand P1, GemmOperand Q1, int np1, int nq1, const int* seg,
                                  int groups, Epi epi, hipStream_t stream) {
  if (np0 <= 0 || nq0 <= 0 || np1 <= 0 || nq1 <= 0 || (np0 | nq0 | np1 | nq1) % 256 || groups <= 0 || groups > 64 || !seg) return TFB_ERR_SHAPE;
  for (const GemmOperand& o : {P0, Q0, P1, Q1}) {
    if (o.ld <= 0 || o.ld > (1L << 28)) return TFB_ERR_SHAPE;
    if (((uintptr_t)o.base | (uintptr_t)o.ld) & 15) return TFB_ERR_ARG;
  }
  const long t0 = (long)(np0 / 256) * (nq0 / 256), t1 = (long)(np1 / 256) * (nq1 / 256);
  if ((t0 + t1) * groups >= (1L << 24)) return TFB_ERR_SHAPE;
  PpArgs a = {};
  a.P = P0;
  a.Q = Q0;
  a.P1 = P1;
  a.Q1 = Q1;
  a.splits = 1;
  a.nout0 = (int)t0;
  a.nout = a.ntiles = (int)(t0 + t1);
  a.ipx = (a.nout + 7) / 8;
  a.nwg = 8 * a.ipx * groups;
  a.p_fast = np0 <= nq0;
  a.nfast = (a.p_fast ? np0 : nq0) / 256;
  a.p_fast1 = np1 <= nq1;
  a.nfast1 = (a.p_fast1 ? np1 : nq1) / 256;
  a.R = a.GW = a.panel = a.gw_last = 1;
  a.d_nfast = fastdiv_make(a.nfast);
  a.d_nfast1 = fastdiv_make(a.nfast1);
  a.d_panel = a.d_gw = a.d_gw_last = fastdiv_make(1);
  a.d_nout = fastdiv_make(a.nout);
  a.d_ipx = fastdiv_make(a.ipx);
  a.seg = seg;
  a.ngroups = groups;
  hipLaunchKernelGGL((gemm_pp_kernel<1, TFB_FMT_E4M3, TFB_FMT_E5M2, TFB_K_STRIDED, TFB_K_STRIDED, Epi>), dim3(a.nwg), dim3(512), 0, stream, a, epi);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}

// A grouped fp8 product over the rows of all groups (row_group: PpArgs), both operands k-contiguous: D[p][q] = sum_k P_g[p][k] Q[q][k]. What it
// leaves is the ring's (gemm_ring_rest).
static inline int gemm_pp_rows_wgs() { return (int)tfb_resident_slots(1) & ~7; }
// Used where half the CUs or more have an output tile (counted by the rows the tables hold). What bounds it is the k-loop, as in dense launches;
// the 128 x 128 kernel moves twice the operand bytes (16384 tokens, two of eight experts, d 1024, F 2816: 120 and 131 -> 88 us, and 16.5 for the rest).
// Forward and backward of the layer, us, 128 x 128 -> this (tiles over CUs): d 1024, F 2816: 6144 tokens x 2 (0.8) 418 -> 405, 16384 x 2 (2.1) 849
// -> 803, 4096 x 2 (0.55) 338 -> 330, 6144 x 1 (0.43) 281 -> 301; d 768, F 1536: 16384 x 2 532 -> 495, 6144 x 2 (0.6) 265 -> 249, 8192 x 1 (0.42) 215 ->
// 217; d 512, F 1024: 16384 x 2 (1.05) 306 -> 299, 8192 x 2 (0.53) 203 -> 200, 12288 x 1 (0.4) 175 -> 189.
static inline bool gemm_pp_rows_applies(long np, long rows, long kbytes) {
  const long cus = gemm_pp_rows_wgs();
  return TFB_PP && cus > 0 && np % 256 == 0 && rows % 128 == 0 && rows <= 128L * 4096 && kbytes % 128 == 0 && kbytes >= 256 && (rows / 128) * (np / 256) >= cus;
}
template <int FMTP, int FMTQ, class Epi>
static int gemm_pp_launch_rows(GemmOperand P, long p_group_stride, GemmOperand Q, int np, long rows, long kbytes, const int* row_group, Epi epi,
                               hipStream_t stream) {
  const int nwg = gemm_pp_rows_wgs();
  if (nwg <= 0 || np <= 0 || np % 256 || rows <= 0 || rows % 128 || rows > 128L * 4096 || kbytes % 128 || kbytes < 256 || !row_group) return TFB_ERR_SHAPE;
  if (P.ld <= 0 || Q.ld <= 0 || P.ld > (1L << 28) || Q.ld > (1L << 28)) return TFB_ERR_SHAPE;
  if (((uintptr_t)P.base | (uintptr_t)Q.base | (uintptr_t)P.ld | (uintptr_t)Q.ld | (uintptr_t)p_group_stride) & 15) return TFB_ERR_ARG;
  PpArgs a = {};
  a.P = P;
  a.Q = Q;
  a.splits = 1;
  a.nk_total = (int)(kbytes / 128);
  a.nfast = np / 256;
  a.d_nfast = fastdiv_make(a.nfast);
  a.nwg = nwg;
  a.row_group = row_group;
  a.row_tiles = (int)(rows / 128);
  a.p_group_stride = p_group_stride;
  hipLaunchKernelGGL((gemm_pp_kernel<1, FMTP, FMTQ, TFB_K_CONTIG, TFB_K_CONTIG, Epi>), dim3(nwg), dim3(512), 0, stream, a, epi);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}
