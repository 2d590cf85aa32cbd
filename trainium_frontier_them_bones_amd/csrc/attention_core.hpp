// What the attention kernels of both head dimensions share: operand views, MFMA and lane helpers, and the rules by which a
// workgroup gets its blocks.
#pragma once
#include <algorithm>
#include "common.hpp"

// dK and dV by pairs of wavefronts (attention_dkdv.hip). Its loads address 32 tokens by a 32-bit offset.
int tfb_attn_dkdv_impl(const void* q, const long* qs, const void* k, const long* ks, const void* v, const long* vs, const void* go,
                       const long* gos, void* dk, const long* dks, void* dv, const long* dvs, const float* stats, int B, int H, int T,
                       int D, float scale, const void* cos_t, const void* sin_t, int nw, hipStream_t s);
static inline bool tfb_attn_dkdv_strides_ok(const long* qs, const long* gos) {
  return qs[2] >= 0 && qs[2] < (1L << 25) && gos[2] >= 0 && gos[2] < (1L << 25);
}

// dQ and the row statistics by pairs of wavefronts, 64 queries a workgroup (attention_dq.hip). The same holds of its loads.
int tfb_attn_dq_pair_impl(const void* q, const long* qs, const void* k, const long* ks, const void* v, const long* vs, const void* o,
                          const long* os, const void* go, const long* gos, void* dq, const long* dqs, const float* lse, float* stats, int B, int H,
                          int T, int D, float scale, const void* cos_t, const void* sin_t, int nw, hipStream_t s);
// The forward by pairs of wavefronts, 64 queries a workgroup (attention_fwd.hip). The same holds of its loads.
int tfb_attn_fwd_pair_impl(const void* q, const long* qs, const void* k, const long* ks, const void* v, const long* vs, void* o, const long* os,
                           float* lse, int B, int H, int T, int D, float scale, int nw, hipStream_t s);
// Pairs divide a block's work between twice the wavefronts and do a little more of it. That shortens a launch whose longest block sets the
// time and not one whose blocks keep the SIMDs busy, so what counts is the work a CU has in units of the longest block. A causal
// block i of nx has i + 1 tiles, a band leaves it nw at most: the blocks of a short sequence or a narrow band are nearly alike and fill the
// chip with half as many as those of a long sequence.
struct AttnLoad {
  long longest, work, blocks;   // tiles of the longest block; of all blocks; how many they are
};
static inline AttnLoad attn_load(int T, long nbh, int nw) {
  const long nx = T / 128, w = nw > 0 && nw < nx ? nw : nx;
  return AttnLoad{w, nbh * (w * (w + 1) / 2 + (nx - w) * w), nbh * nx};
}
// dQ: half a block for each CU (its workgroups of 64 queries are twice the blocks and then have a CU each), or as much work as the line
// below (D = 128 has one such workgroup on a CU, D = 64 two). dQ and dK/dV, us, one wavefront to 32 queries -> pairs, blocks in brackets:
//   D = 64   T128 [128] 14.6 -> 14.5, [160] 14.8 -> 16.3; T256 [128] 20.0 -> 19.2, [192] 20.5 -> 21.1; T512 [192] 28.5 -> 27.8, [288] 30.5 -> 31.9;
//            T1024 [288] 46.1 -> 43.2, [384] 47.9 -> 50.6; T2048 [384] 80.6 -> 79.7, [512] 87.2 -> 88.8; T4096 [384] 147 -> 139, [576] 168 -> 172;
//            bands: 1 T2048 [192] 15.8 -> 17.1; 2 T2048 [128] 20.2 -> 19.3, [192] 21.0 -> 22.7; 4 T1024 [128] 28.4 -> 26.2, [256] 29.3 -> 30.8;
//            8 T2048 [192] 44.2 -> 43.2, [320] 49.1 -> 52.6
//   D = 128  T128 [128] 25.1 -> 23.5, [192] 27.1 -> 31.4; T256 [128] 30.9 -> 28.1, [192] 32.5 -> 34.8; T512 [160] 42.0 -> 40.3, [288] 49.9 -> 55.5;
//            T1024 [256] 65.4 -> 60.8, [320] 69.9 -> 74.6; T2048 [288] 112 -> 110, [384] 120 -> 124; T4096 [320] 207 -> 198, [448] 234 -> 245;
//            bands: 1 T2048 [192] 28.7 -> 32.9; 4 T1024 [128] 41.8 -> 36.7, [192] 43.1 -> 47.1; 8 T2048 [128] 62.7 -> 52.9, [256] 67.0 -> 73.7
static inline bool tfb_attn_dq_pair_applies(int D, int T, long nbh, int nw, const long* ks, const long* vs) {
  const AttnLoad l = attn_load(T, nbh, nw);
  const long cus = tfb_resident_slots(1), line = D == 64 ? std::min(l.longest + 7, 16L) : std::min(l.longest + 7, 17L);
  return (2 * l.blocks <= cus || (D == 64 ? 20 : 26) * l.work <= line * cus * l.longest) && tfb_attn_dkdv_strides_ok(ks, vs);
}
// dK/dV at D = 64 (a workgroup of eight wavefronts on a CU, in place of one or two of four): one block for each CU, or as much work as this line,
// but not where every block is one tile. dQ and dK/dV, us, one or two workgroups of four -> pairs:
//   T128 [64] 14.0 -> 15.3; T256 [192] 20.5 -> 20.3, [288] 25.1 -> 27.7; T512 [256] 29.1 -> 27.6, [320] 31.0 -> 32.3;
//   T1024 [384] 47.9 -> 46.4, [448] 50.0 -> 51.4; T2048 [512] 87.2 -> 82.2, [576] 91.2 -> 98.0; T4096 [512] 160 -> 146, [576] 168 -> 169; bands:
//   1 T2048 [128] 14.6 -> 15.8; 2 T2048 [256] 22.0 -> 21.6, [320] 30.9 -> 35.6; 4 T2048 [256] 29.8 -> 28.1, [320] 42.6 -> 46.2;
//   8 T2048 [256] 45.5 -> 41.0, [320] 49.1 -> 51.9
static inline bool tfb_attn_dkdv_pair_applies(int T, long nbh, int nw, const long* qs, const long* gos) {
  const AttnLoad l = attn_load(T, nbh, nw);
  const long cus = tfb_resident_slots(1);
  return l.longest > 1 && (l.blocks <= cus || 32 * l.work <= std::min(l.longest + 20, 36L) * cus * l.longest) && tfb_attn_dkdv_strides_ok(qs, gos);
}
// dK/dV by pairs with 64 keys a workgroup in place of 128: the longest block is half as long, what a block does besides its loop counts twice. One
// workgroup for each CU always; beyond, by the work a CU has in units of the longest block of 128, as above: at D = 64 two workgroups share a CU,
// at D = 128 (141 KB of LDS) one has it alone. dQ and dK/dV, us, 128 keys -> 64, blocks of 128 in brackets:
//   D = 64   T128 [128] 13.7 -> 12.8, [192] 14.8 -> 15.1; T256 [128] 18.1 -> 15.2, [256] 20.2 -> 18.4, [320] 23.9 -> 24.7; T512 [192] 24.7 -> 21.4,
//            [320] 29.1 -> 27.9, [384] 30.3 -> 30.5; T1024 [256] 36.4 -> 32.7, [384] 44.9 -> 41.3, [512] 48.0 -> 47.8; T2048 [192] 55.1 -> 48.3, [384] 67.7 ->
//            66.4, [512] 80.1 -> 79.7, [576] 90.4 -> 91.0; T4096 [256] 100.3 -> 91.7, [384] 119 -> 117, [448] 136 -> 137; bands: 1 T2048 [128] 13.3 -> 12.4,
//            [192] 15.0 -> 15.0; 2 [256] 20.9 -> 19.6, [384] 30.7 -> 29.7; 4 [256] 27.3 -> 26.1, [384] 42.7 -> 39.8; 8 [192] 36.9 -> 33.2, [256] 39.8 -> 40.0
//   D = 128  T128 [128] 21.7 -> 18.6, [192] 25.6 -> 27.4; T256 [128] 27.9 -> 23.8, [192] 32.3 -> 32.4; T512 [192] 42.0 -> 40.9, [256] 43.0 -> 43.9;
//            T1024 [192] 55.6 -> 50.0, [320] 68.2 -> 75.3; T1664 [208] 74.7 -> 66.0, [260] 89.3 -> 90.0; T2048 [256] 93.7 -> 88.4, [320] 114 -> 122; T4096 [256]
//            162 -> 150, [320] 201 -> 210; bands of T2048: 1 [128] 21.8 -> 18.4, [192] 28.6 -> 30.1; 4 [128] 36.0 -> 31.5, [192] 44.4 -> 51.0
static inline bool tfb_attn_dkdv_half_applies(int D, int T, long nbh, int nw, const long* qs, const long* gos) {
  if (!tfb_attn_dkdv_strides_ok(qs, gos)) return false;
  const AttnLoad l = attn_load(T, nbh, nw);
  const long cus = tfb_resident_slots(1), nx = T / 128;
  if (2 * l.blocks <= cus) return true;
  if (D == 128) return 1000 * l.work <= 535 * cus * l.longest;
  if (l.longest == 1) return false;
  const long line = l.longest <= 4 && 4 * l.longest <= nx ? 14 : l.longest == nx && nx >= 8 && nx <= 16 ? 10 : 8;
  return 10 * l.work <= line * cus * l.longest;
}

// The forward: one workgroup of 64 queries for each CU (but for blocks of one tile of D = 128), or as much work as this line, in the same units.
// At D = 128 a second workgroup finds no room on a CU, so beyond one for each only a sequence pays whose light blocks end early enough for the
// rest: six tiles and more without a band. us, one wavefront to 32 queries -> pairs, blocks in brackets:
//   D = 64   T128 [128] 5.9 -> 5.4, [192] 6.1 -> 6.2; T256 [192] 7.5 -> 6.7, [320] 9.9 -> 9.9; T512 [192] 9.8 -> 8.8, [256] 10.0 -> 9.2, [320] 11.1 -> 12.0; T1024
//            [256] 14.8 -> 13.4, [320] 15.3 -> 15.7; T1664 [312] 21.2 -> 19.5, [364] 21.5 -> 22.8; T2048 [192] 24.2 -> 21.2, [320] 24.8 -> 22.8, [384] 25.2 ->
//            27.1; T4096 [320] 44.7 -> 40.1, [384] 45.3 -> 47.1; bands of T2048: 2 [128] 7.0 -> 6.2, [192] 7.3 -> 7.4; 4 [128] 9.4 -> 8.3, [192] 9.8 -> 10.6;
//            8 [192] 14.8 -> 13.6, [256] 15.2 -> 17.2
//   D = 128  T128 [96] 7.8 -> 7.7, [144] 8.0 -> 11.3; T256 [128] 9.5 -> 9.2, [144] 9.8 -> 11.5; T384 [108] 11.1 -> 10.4, [144] 11.5 -> 12.6; T512 [96] 12.7 ->
//            11.8, [144] 13.4 -> 13.3, [192] 13.4 -> 15.8; T640 [120] 14.6 -> 13.4, [180] 15.1 -> 16.1; T768 [144] 16.4 -> 15.4, [216] 16.8 -> 19.2; T1024 [128]
//            19.3 -> 18.2, [192] 19.7 -> 19.6, [224] 20.6 -> 22.6; T1664 [208] 27.5 -> 25.8, [260] 28.9 -> 35.4; T2048 [192] 32.4 -> 31.2, [256] 32.8 -> 34.3;
//            T4096 [192] 58.1 -> 54.5, [256] 58.2 -> 57.7; bands: 2 T2048 [128] 9.6 -> 9.2, [192] 10.4 -> 16.3; 4 T2048 [128] 12.7 -> 12.1, [192] 13.5 -> 21.5;
//            8 T2048 [128] 19.3 -> 18.2, [192] 19.9 -> 27.3
static inline bool tfb_attn_fwd_pair_applies(int D, int T, long nbh, int nw, const long* ks, const long* vs) {
  const AttnLoad l = attn_load(T, nbh, nw);
  const long cus = tfb_resident_slots(1), nx = T / 128;
  if (!tfb_attn_dkdv_strides_ok(ks, vs) || (D == 128 && l.longest == 1)) return false;
  if (2 * l.blocks <= cus) return true;
  if (D == 64) return 1000 * l.work <= 665 * cus * l.longest;
  return l.longest == nx && nx >= 6 && 1000 * l.work <= (nx >= 8 ? 440 : 350) * cus * l.longest;
}

namespace {

struct AttnT {
  bf16_t* p;
  long sb, sh, st;
};
AttnT mk(const void* p, const long* s) { return AttnT{(bf16_t*)p, s[0], s[1], s[2]}; }

typedef __attribute__((address_space(3))) void lds_void_t;
typedef const __attribute__((address_space(1))) void glb_void_t;

constexpr float LOG2E = 1.4426950408889634f;
constexpr float LN2 = 0.6931471805599453f;

__device__ __forceinline__ f32x16 mfma_bf16(bf16x8 a, bf16x8 b, f32x16 c) {
  return __builtin_amdgcn_mfma_f32_32x32x16_bf16(a, b, c, 0, 0, 0);
}
__device__ __forceinline__ float fast_exp2(float x) { return __builtin_amdgcn_exp2f(x); }
__device__ __forceinline__ bf16x8 frag_from(uint32_t a, uint32_t b, uint32_t c, uint32_t d) {
  u32x4 v = {a, b, c, d};
  return __builtin_bit_cast(bf16x8, v);
}
__device__ __forceinline__ float max_halves(float x) {  // the larger of the two lanes' that share a query
  float y = x;
  asm volatile("s_nop 1\n\tv_permlane32_swap_b32 %0, %1" : "+v"(x), "+v"(y));
  return fmaxf(x, y);
}

// Store one token's gradient row from the two 32-element halves a lane's accumulators hold (elements 8 j + 4 lh + i of
// each half), scaled and rounded once to bf16; with cos / sin tables ([T][32] bf16) the inverse RoPE rotation
// (y1 = x1 c - x2 s, y2 = x2 c + x1 s on the rounded values, rounded again: what a separate pass over the bf16
// gradient computes) is applied on the way out.
__device__ __forceinline__ void store_grad_row(const f32x16 (&acc)[2], float scale, bf16_t* row, const bf16_t* cs,
                                               const bf16_t* sn, int tok, int lh) {
#pragma unroll
  for (int j = 0; j < 4; ++j) {
    const int d = 8 * j + 4 * lh;
    u32x2 w1 = {pack2bf(acc[0][4 * j] * scale, acc[0][4 * j + 1] * scale),
                pack2bf(acc[0][4 * j + 2] * scale, acc[0][4 * j + 3] * scale)};
    u32x2 w2 = {pack2bf(acc[1][4 * j] * scale, acc[1][4 * j + 1] * scale),
                pack2bf(acc[1][4 * j + 2] * scale, acc[1][4 * j + 3] * scale)};
    if (cs) {
      const u32x2 c = *(const u32x2*)(cs + (long)tok * 32 + d), s = *(const u32x2*)(sn + (long)tok * 32 + d);
      u32x2 o1, o2;
#pragma unroll
      for (int x = 0; x < 2; ++x) {
        const float a0 = bflo(w1[x]), a1 = bfhi(w1[x]), b0 = bflo(w2[x]), b1 = bfhi(w2[x]);
        const float c0 = bflo(c[x]), c1 = bfhi(c[x]), s0 = -bflo(s[x]), s1 = -bfhi(s[x]);
        o1[x] = pack2bf(a0 * c0 + b0 * s0, a1 * c1 + b1 * s1);
        o2[x] = pack2bf(b0 * c0 - a0 * s0, b1 * c1 - a1 * s1);
      }
      w1 = o1;
      w2 = o2;
    }
    *(u32x2*)(row + d) = w1;
    *(u32x2*)(row + 32 + d) = w2;
  }
}

// Workgroup -> (block along the sequence, batch*head): consecutive workgroup ids are dealt round-robin to the 8 XCDs, each with its own
// L2, so the ids are re-dealt to keep all sequence blocks of one (batch, head) - which stream the same K/V (or Q/dO) tiles - on one
// XCD. With one block per workgroup (gridDim.x = nx) the order is slot-major, the heaviest block of each pair first: workgroups start in
// id order, and the causal blocks differ in work by a factor of nx. That order matters more than the XCD: where the pairs are no
// multiple of 8 and cannot be dealt to the XCDs evenly, it is kept without that (pair by pair in order, the last pairs' heavy blocks
// ran on alone; T2048 D64 12 heads B3 forward 57 -> 34 us, backward 165 -> 96; B7 103 -> 73, 297 -> 195; T3072 D128 6 heads B2
// 64 -> 52, 230 -> 174). nx = blocks per (batch, head), nbh = batch*head count. One division and no branch: behind branches the kernels'
// other arguments were loaded only after it (forward, us: D128 T2048 4 heads 32.6 -> 31.6, 12 heads 34.3 -> 33.3; D64 T256 12 heads 7.1 -> 6.9).
// turn: the workgroups that start first, one on a CU, where a second will share it with some of them (0: none does). These run in the opposite
// order, so that the second ones, the shortest, come to the shorter of them and not to the longest (us: forward D128 T1664 24 heads 31.9 -> 29.6,
// D64 T2048 24 heads 29.1 -> 27.0; dQ and dK/dV of 12 heads 62.1 -> 60.0, with 64 keys a workgroup 55.6 -> 52.8).
__device__ __forceinline__ void xcd_block(int nx, int nbh, int& bx, int& bh, int turn = 0) {
  const int gx = gridDim.x;
  int lin = blockIdx.y * gx + blockIdx.x;
  const int xcd = lin & 7;
  if (lin < turn) lin = turn - 8 - lin + 2 * xcd;   // (a multiple of 8: the XCD stays)
  const bool dealt = nbh % 8 == 0, single = gx == nx;
  const unsigned id = dealt ? lin >> 3 : lin, by = single ? (dealt ? nbh >> 3 : nbh) : gx;
  const int quot = (int)(id / by), rem = (int)(id - quot * by);
  bx = single ? quot : rem;
  bh = single ? rem : quot;
  bh = dealt ? xcd + 8 * bh : bh;
}

// Causal work per 128-token block grows linearly along the sequence, and workgroups are dispatched in id order: with one
// block per workgroup the heaviest blocks of the last (batch, head) pairs start when most of the grid has drained and
// run on alone (for 16 blocks x 192 pairs on 512 slots: 17 % of the kernel's time). When the block count nx is even a
// workgroup therefore does block i and then block nx - 1 - i (gridDim.x = nx / 2): every workgroup carries the same
// work. `heavy_last` = the work grows with the block index (query blocks) rather than falls (key blocks); the heavier
// block of the pair runs first either way.
__device__ __forceinline__ int paired_passes(int nx) { return (int)gridDim.x * 2 == nx ? 2 : 1; }
__device__ __forceinline__ int paired_block(int nx, int bx, int pass, bool heavy_last) {
  const int first = heavy_last ? nx - 1 - bx : bx;
  return pass == 0 ? first : nx - 1 - first;
}
// First 64-key tile a 128-token query tile qb sees under a band of nw key tiles (a query of tile i sees the keys k <= q
// of tiles i - nw + 1 .. i: band_mask, round2/source/kernels/nki_attn_bandpro.py:1654); 0 without a band (nw <= 0).
__device__ __forceinline__ int band_first_tile(int qb, int nw) { return nw > 0 && qb - nw + 1 > 0 ? 2 * (qb - nw + 1) : 0; }
// Blocks are paired when the paired grid fills its rounds of resident workgroups to 90 % (or is long enough not to care); otherwise
// one block per workgroup, the heaviest first (B8 H8 T512 forward 14.3 -> 10.8 us, backward 43 -> 33; B1 H12 T2048 31 -> 27, 89 -> 80).
__host__ inline unsigned paired_grid(int nx, int nbh, int per_cu) {
  if (nx % 2) return (unsigned)nx;
  const long wgs = (long)(nx / 2) * nbh, slots = tfb_resident_slots(per_cu), rounds = (wgs + slots - 1) / slots;
  return (unsigned)(wgs * 10 >= rounds * slots * 9 ? nx / 2 : nx);
}

// xcd_block's turn for nx x nbh workgroups of which two share a CU, blocks paired by paired_grid(nx, nbh, 2) or one by one
__host__ inline int first_round(int nx, int nbh, bool may_pair) {
  const int cus = (int)tfb_resident_slots(1) & ~7;
  return (long)nx * nbh > cus && !(may_pair && (int)paired_grid(nx, nbh, 2) != nx) ? cus : 0;
}

}  // namespace
