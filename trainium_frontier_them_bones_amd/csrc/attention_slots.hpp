// Tiles, fragments and slots of the attention kernels' hand-placed loops: how a 64-token tile lies in LDS, the loads that bring it there,
// and the fragment reads.
#pragma once
#include <type_traits>

#include "attention_core.hpp"

namespace {

typedef __attribute__((address_space(1))) uint8_t glb_u8_t;

template <int D>
struct Geo {
  static constexpr int ROWB = 2 * D;        // bytes of a token's row
  static constexpr int TILE = 64 * ROWB;    // bytes of a 64-token tile
  static constexpr int NKS = D / 16;        // MFMA k-steps over the head dimension
  static constexpr int NDT = D / 32;        // 32-element tiles of the head dimension
  static constexpr int LPT = ROWB / 16;     // lanes (16-byte chunks) per token
  static constexpr int TPI = 64 / LPT;      // tokens per 1 KB load instruction
  // slot swizzle: chunk c of token t at slot c ^ swz(t)
  __device__ static __forceinline__ int swz(int t) {
    if (D == 64) return (((t >> 1) & 1) << 2) | ((t >> 2) & 3);
    return ((t & 3) << 2) | ((t >> 2) & 3);
  }
};

// This wavefront's share of a (16 NI TPI / 4 ...)-token tile load: instructions g = wave + 4 i, i < NI, each TPI tokens.
template <int D, int NI>
struct TileLoad {
  typedef Geo<D> G;
  uint32_t voff;
  int wave;
  __device__ __forceinline__ void init(long stride, int wave_, int lane) {
    wave = wave_;
    const int lrow = lane / G::LPT;
    // token = TPI g + lrow with g = wave + 4 i: the swizzle depends on g only through bits that 4 i does not touch
    const int chunk = (lane % G::LPT) ^ G::swz(G::TPI * wave + lrow);
    voff = (uint32_t)((G::TPI * wave + lrow) * stride + chunk * 16);
  }
  __device__ __forceinline__ void issue_one(int i, const uint8_t* rows, long stride, uint8_t* lds) const {
    const glb_u8_t* r = (const glb_u8_t*)rows;
    uint32_t o = voff;
    asm volatile("" : "+v"(o));   // (its widening stays in this block, where the load takes it as a 32-bit offset)
    __builtin_amdgcn_global_load_lds((glb_void_t*)(r + i * (4 * G::TPI) * stride + o), (lds_void_t*)(lds + (wave + 4 * i) * 1024), 16, 0, 0);
  }
  __device__ __forceinline__ void issue(const uint8_t* rows, long stride, uint8_t* lds) const {
    const glb_u8_t* r = (const glb_u8_t*)rows;   // (uniform base + 32-bit lane offset: no 64-bit address per lane)
#pragma unroll
    for (int i = 0; i < NI; ++i) {
      __builtin_amdgcn_global_load_lds((glb_void_t*)(r + voff), (lds_void_t*)(lds + (wave + 4 * i) * 1024), 16, 0, 0);
      r += 4 * G::TPI * stride;
    }
  }
};

// One token's gradient row from the NDT accumulators a lane holds (elements 32 dt + 8 j + 4 lh + i), scaled and rounded
// once to bf16.
template <int D>
__device__ __forceinline__ void store_grad_row(const f32x16 (&acc)[Geo<D>::NDT], float scale, bf16_t* row, int lh) {
#pragma unroll
  for (int dt = 0; dt < Geo<D>::NDT; ++dt)
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      u32x2 w = {pack2bf(acc[dt][4 * j] * scale, acc[dt][4 * j + 1] * scale),
                 pack2bf(acc[dt][4 * j + 2] * scale, acc[dt][4 * j + 3] * scale)};
      *(u32x2*)(row + 32 * dt + 8 * j + 4 * lh) = w;
    }
}

// ------------------------------------------------------------------------------------ pipelined fragment reads
// The tile loops below are written slot by slot: one MFMA, the LDS read of the fragment that a later slot needs, and this slot's
// share of the elementwise work, kept in that order by sched_barrier(0). Fragments are read by inline assembly and tied to an
// explicit s_waitcnt lgkmcnt(n) right before their MFMA: left to the compiler, each read sits in front of its MFMA and every one
// pays the LDS latency.
typedef int i32x4_t __attribute__((ext_vector_type(4)));

template <int I, int N, class F>
__device__ __forceinline__ void slots(F&& f) {
  if constexpr (I < N) {
    f(std::integral_constant<int, I>{});
    slots<I + 1, N>(f);
  }
}
__device__ __forceinline__ void slot_end() { __builtin_amdgcn_sched_barrier(0); }

// values made in this slot (they would otherwise sink to the block that uses them)
__device__ __forceinline__ void pin(float& a, float& b) { asm volatile("" : "+v"(a), "+v"(b)); }
template <class T>
__device__ __forceinline__ void pin(T& a) { asm volatile("" : "+v"(a)); }
__device__ __forceinline__ int opaque(int x) {  // (comparisons against it stay where they are used, not in registers across the loop)
  asm volatile("" : "+v"(x));
  return x;
}
struct RowFrag {  // a token-major fragment on its way: one 16-byte read
  i32x4_t v;
  template <int OFF>
  __device__ __forceinline__ void request(uint32_t addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v) : "v"(addr), "n"(OFF));
  }
  __device__ __forceinline__ bf16x8 get() const { return __builtin_bit_cast(bf16x8, v); }
};
struct ColFrag {  // a transposed fragment: two 8-byte reads
  u32x2 a, b;
  template <int OFF>
  __device__ __forceinline__ void request(uint32_t lo, uint32_t hi) {
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(a) : "v"(lo), "n"(OFF));
    asm volatile("ds_read_b64_tr_b16 %0, %1 offset:%2" : "=v"(b) : "v"(hi), "n"(OFF));
  }
  __device__ __forceinline__ bf16x8 get() const { return frag_from(a.x, a.y, b.x, b.y); }
};
// Two fragments are waited for together: one wavefront alone on its SIMD issues an instruction every five cycles, seven under an MFMA.
// AFTER: LDS instructions issued since the second's.
template <int AFTER>
__device__ __forceinline__ void landed(RowFrag& x, RowFrag& y) {
  asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(x.v), "+v"(y.v) : "n"(AFTER));
}
template <int AFTER>
__device__ __forceinline__ void landed(ColFrag& x, ColFrag& y) {
  asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(x.a), "+v"(x.b), "+v"(y.a), "+v"(y.b) : "n"(AFTER));
}
// Per-lane addresses of the fragments of a tile at `base`. Token-major, rows[s]: token lane & 31, elements 16 s + 8 (lane >> 5) .. + 7.
// Transposed, lo[dt] and hi[dt]: element (MFMA row) 32 dt + (lane & 31), tokens 4 lh + {0..3} and 8 + 4 lh + {0..3}. A tile's place,
// the 32-token half and the 16-token step are added, as the instruction's offset where they are constants.
template <int D>
struct FragAddr {
  uint32_t rows[Geo<D>::NKS], lo[Geo<D>::NDT], hi[Geo<D>::NDT];
  __device__ __forceinline__ void init(uint32_t base, int lane) {
    typedef Geo<D> G;
    const int lr = lane & 31, lh = lane >> 5, g4 = lane >> 4, j = lane & 15;
#pragma unroll
    for (int s = 0; s < G::NKS; ++s) rows[s] = base + lr * G::ROWB + (((2 * s + lh) ^ G::swz(lr)) << 4);
    const int t = 4 * (g4 >> 1) + (j >> 2);
#pragma unroll
    for (int dt = 0; dt < G::NDT; ++dt) {
      const int d = 32 * dt + 16 * (g4 & 1) + 4 * (j & 3);
      lo[dt] = base + t * G::ROWB + (((d >> 3) ^ G::swz(t)) << 4) + ((d & 4) << 1);
      hi[dt] = base + (t + 8) * G::ROWB + (((d >> 3) ^ G::swz(t + 8)) << 4) + ((d & 4) << 1);
    }
  }
};
// all of this wavefront's loads into LDS have landed, and every wavefront is here
__device__ __forceinline__ void tile_barrier() { asm volatile("s_waitcnt vmcnt(0)\n\ts_barrier" ::: "memory"); }

struct StatFrag {  // 32 rows' statistics as an accumulator's start: four 16-byte reads
  f32x4 v[4];
  template <int OFF>
  __device__ __forceinline__ void request(uint32_t addr) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v[0]) : "v"(addr), "n"(OFF));
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v[1]) : "v"(addr), "n"(OFF + 32));
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v[2]) : "v"(addr), "n"(OFF + 64));
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v[3]) : "v"(addr), "n"(OFF + 96));
  }
  template <int AFTER>
  __device__ __forceinline__ void landed(f32x16& x) {
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]) : "n"(AFTER));
#pragma unroll
    for (int e = 0; e < 16; ++e) x[e] = v[e >> 2][e & 3];
  }
};

}  // namespace
