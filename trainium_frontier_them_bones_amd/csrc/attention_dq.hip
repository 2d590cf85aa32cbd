// dQ of causal flash attention on gfx950 for launches that do not fill the chip: 64 queries per workgroup, two wavefronts to every 32.
//
// With one wavefront to 32 queries the longest block sets such a launch's time, and a wavefront alone on its SIMD takes all of its
// instructions in turn. Here each of a pair makes S, P, dP and dS of one 32-key half of a tile, hands dS to the other through LDS and adds
// both halves' dS K to its own half of dQ's columns: half the instructions a tile, twice the wavefronts. Every sum is made by one wavefront in
// the order of the kernels with one: the same bits.
// What bounds it: instructions, 186 a tile at D = 64 and 315 at D = 128 with 12 and 24 MFMAs among them, one every 5.7 to 6 cycles, and a
// barrier a tile; with S and dP made one tile further ahead, or columns and rows in turn, a tile takes as long. us, one wavefront to 32
// queries -> this: D = 64 B1 H12 T2048 35.1 -> 28.2, B1 H2 T8192 112 -> 77; D = 128 B1 H8 T2048 54.8 -> 36.4, B3 H4 T384 18.8 -> 13.2.
#include "attention_slots.hpp"

namespace {

struct DsTile {  // dS of 32 queries and 64 keys, packed: fragment i is the operand of the 16 keys i
  u32x4 v[4];
  __device__ __forceinline__ void request(uint32_t at) {
    asm volatile("ds_read_b128 %0, %1" : "=v"(v[0]) : "v"(at));
    asm volatile("ds_read_b128 %0, %1 offset:1024" : "=v"(v[1]) : "v"(at));
    asm volatile("ds_read_b128 %0, %1 offset:2048" : "=v"(v[2]) : "v"(at));
    asm volatile("ds_read_b128 %0, %1 offset:3072" : "=v"(v[3]) : "v"(at));
  }
  template <int AFTER>
  __device__ __forceinline__ void landed() {
    asm volatile("s_waitcnt lgkmcnt(%4)" : "+v"(v[0]), "+v"(v[1]), "+v"(v[2]), "+v"(v[3]) : "n"(AFTER));
  }
};

template <int D>
__global__ __launch_bounds__(256, 2) void attn_dq_pair_kernel(AttnT q, AttnT k, AttnT v, AttnT go, AttnT dq, float* __restrict__ stats, long rows,
                                                              int T, int H, float scale, float sl2, const bf16_t* __restrict__ cs,
                                                              const bf16_t* __restrict__ sn, int nw, AttnT o, const float* __restrict__ lse, int turn) {
  typedef Geo<D> G;
  constexpr int TILE = G::TILE, NKS = G::NKS, NDT = G::NDT, MDT = NDT / 2;  // MDT: 32-column tiles of dQ that are this wavefront's
  constexpr int AH = 4, NL = 16 / G::TPI;     // items asked for ahead of their use; load instructions of a wavefront for a K or V tile
  constexpr int STAGE = 2 * TILE, XCH = 4 * STAGE;  // four stages of a K and a V tile; then dS: two tiles of two pairs of two halves
  constexpr int NP = 2 * NKS;                 // items of a tile: K and V rows, dS (item NP), K columns
  __shared__ __attribute__((aligned(1024))) uint8_t lds[XCH + 2 * 8192];
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), pair = wave >> 1, half = wave & 1;
  const int nx = T / 64;
  int bx, bh;
  xcd_block(nx, gridDim.y, bx, bh, turn);
  const int b = bh / H, h = bh % H, qb = nx - 1 - bx;   // the most tiles first
  const int myq = qb * 64 + pair * 32 + lr;
  const int n = qb + 1, t0 = band_first_tile(qb >> 1, nw);  // tile n - 1 is over the workgroup's own tokens
  const long kst = k.st * 2, vst = v.st * 2;
  const uint8_t* kp = (const uint8_t*)(k.p + b * k.sb + h * k.sh);
  const uint8_t* vp = (const uint8_t*)(v.p + b * v.sb + h * v.sh);
  TileLoad<D, NL> lk, lv;
  lk.init(kst, wave, lane);
  lv.init(vst, wave, lane);
  // A tile's loads one by one, tile after tile from t0 on (past the last: that one again, into a stage nobody reads)
  const uint8_t *kl = kp + (long)t0 * 64 * kst, *vl = vp + (long)t0 * 64 * vst;
  auto load_one = [&](int tile, int i) __attribute__((always_inline)) {
    uint8_t* to = lds + (tile & 3) * STAGE;
    if (i < NL) lk.issue_one(i, kl, kst, to);
    else lv.issue_one(i - NL, vl, vst, to + TILE);
    if (i == 2 * NL - 1 && tile + 1 < n) {
      kl += 64 * kst;
      vl += 64 * vst;
    }
  };

  bf16x8 qf[NKS], gf[NKS];
  {
    const bf16_t* qr = q.p + b * q.sb + h * q.sh + (long)myq * q.st;
    const bf16_t* gr = go.p + b * go.sb + h * go.sh + (long)myq * go.st;
#pragma unroll
    for (int s = 0; s < NKS; ++s) {
      qf[s] = *(const bf16x8*)(qr + 16 * s + 8 * lh);
      gf[s] = *(const bf16x8*)(gr + 16 * s + 8 * lh);
    }
  }
  // the row statistics, left for the dK/dV kernel: -sum_d dO O and -lse / scale
  float myD, myL;
  {
    const bf16_t* orow = o.p + b * o.sb + h * o.sh + (long)myq * o.st;
    float dot = 0.f;
#pragma unroll
    for (int s = 0; s < NKS; ++s) {
      const u32x4 ov = *(const u32x4*)(orow + 16 * s + 8 * lh);
      const u32x4 gv = __builtin_bit_cast(u32x4, gf[s]);
#pragma unroll
      for (int x = 0; x < 4; ++x) {
        dot += bflo(ov[x]) * bflo(gv[x]);
        dot += bfhi(ov[x]) * bfhi(gv[x]);
      }
    }
    dot += __shfl_xor(dot, 32, 64);
    myD = -dot;
    myL = -lse[(long)bh * T + myq] * (1.0f / scale);
  }
#pragma unroll
  for (int t = 0; t < 3; ++t)
#pragma unroll
    for (int i = 0; i < 2 * NL; ++i) load_one(t0 + t, i);

  f32x16 acc[MDT];
#pragma unroll
  for (int i = 0; i < MDT; ++i)
#pragma unroll
    for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;

  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void_t*)lds;
  FragAddr<D> fa;
  fa.init(lds0, lane);
  uint32_t cl[MDT], ch[MDT];
#pragma unroll
  for (int i = 0; i < MDT; ++i) {
    cl[i] = half ? fa.lo[MDT + i] : fa.lo[i];
    ch[i] = half ? fa.hi[MDT + i] : fa.hi[i];
  }
#pragma unroll
  for (int s = 0; s < NKS; ++s) fa.rows[s] += half * (TILE / 2);
  const uint32_t xa = lds0 + XCH + pair * 4096 + lane * 16;

  f32x16 S, dP;
  uint32_t pw[8], xw[8];
  DsTile ds;
  RowFrag rf[2 * NKS];
  ColFrag cf[NKS];
  uint32_t ra[NKS], la[MDT], ha[MDT], xg;
  auto addresses = [&](int row_tile, int col_tile) __attribute__((always_inline)) {
    const uint32_t r = (row_tile & 3) * STAGE, c = (col_tile & 3) * STAGE;
#pragma unroll
    for (int s = 0; s < NKS; ++s) ra[s] = fa.rows[s] + r;
#pragma unroll
    for (int i = 0; i < MDT; ++i) {
      la[i] = cl[i] + c;
      ha[i] = ch[i] + c;
    }
    xg = xa + (col_tile & 1) * 8192;
  };
  auto ask_row = [&](auto item) __attribute__((always_inline)) {
    constexpr int i = decltype(item)::value;
    rf[i].template request<(i / NKS) * TILE>(ra[i % NKS]);
  };
  auto ask_col = [&](auto item) __attribute__((always_inline)) {  // fragment MDT * (16-key step of the tile) + column tile
    constexpr int i = decltype(item)::value;
    cf[i].template request<(i / MDT) * 16 * G::ROWB>(la[i % MDT], ha[i % MDT]);
  };
  auto ask_ds = [&]() __attribute__((always_inline)) { ds.request(xg); };
  auto row_mfma = [&](auto item) __attribute__((always_inline)) {
    constexpr int i = decltype(item)::value;
    if constexpr (i < NKS) S = mfma_bf16(rf[i].get(), qf[i], S);
    else dP = mfma_bf16(rf[i].get(), gf[i - NKS], dP);
  };
  auto col_mfma = [&](auto item) __attribute__((always_inline)) {
    constexpr int i = decltype(item)::value;
    acc[i % MDT] = mfma_bf16(cf[i].get(), __builtin_bit_cast(bf16x8, ds.v[i / MDT]), acc[i % MDT]);
  };
  auto start = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int e = 0; e < 16; ++e) {
      S[e] = myL;
      dP[e] = myD;
    }
  };
  auto p_word = [&](auto word) __attribute__((always_inline)) {
    constexpr int x = decltype(word)::value;
    const float a = fast_exp2(S[2 * x] * sl2), c = fast_exp2(S[2 * x + 1] * sl2);
    pw[x] = pack2bf(a, c);
    pin(pw[x]);
  };
  auto ds_word = [&](auto word) __attribute__((always_inline)) {  // the reference multiplies dP - delta by the rounded P
    constexpr int x = decltype(word)::value;
    xw[x] = pack2bf(bflo(pw[x]) * dP[2 * x], bfhi(pw[x]) * dP[2 * x + 1]);
    pin(xw[x]);
  };
  auto put = [&](int tile) __attribute__((always_inline)) {
    const uint32_t at = xa + (tile & 1) * 8192 + half * 2048;
    const u32x4 lo = {xw[0], xw[1], xw[2], xw[3]}, hi = {xw[4], xw[5], xw[6], xw[7]};
    asm volatile("ds_write_b128 %0, %1\n\tds_write_b128 %0, %2 offset:1024" ::"v"(at), "v"(lo), "v"(hi) : "memory");
  };
  // In front of step t: every wavefront's dS of tile t is in LDS and tile t + 1 has landed; tile t - 1's stage is free.
  auto begin = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)\n\ts_barrier" ::"n"(2 * NL) : "memory"); };

  // A step's parts by themselves, in front of the loop and behind it
  auto rows_of = [&](int tile) __attribute__((always_inline)) {
    addresses(tile, tile);
    slots<0, 2 * NKS>([&](auto i) { ask_row(i); });
    start();
    slots<0, NKS>([&](auto i) { landed<0>(rf[2 * decltype(i)::value], rf[2 * decltype(i)::value + 1]); });
    slots<0, 2 * NKS>([&](auto i) { row_mfma(i); });
    if (tile == n - 1 && half == pair) {
      const int kbase = half * 32 + lh * 4 - pair * 32 - lr;  // key - query of element e is kbase + (e >> 2) * 8 + (e & 3)
#pragma unroll
      for (int e = 0; e < 16; ++e) S[e] = (kbase + (e >> 2) * 8 + (e & 3) > 0) ? -INFINITY : S[e];
    }
    slots<0, 8>([&](auto i) {
      p_word(i);
      ds_word(i);
    });
    put(tile);
  };
  auto cols_of = [&](int tile) __attribute__((always_inline)) {
    addresses(tile, tile);
    ask_ds();
    slots<0, NKS>([&](auto i) { ask_col(i); });
    ds.template landed<0>();
    slots<0, NKS / 2>([&](auto i) { landed<0>(cf[2 * decltype(i)::value], cf[2 * decltype(i)::value + 1]); });
    slots<0, NKS / 2>([&](auto i) { col_mfma(i); });
    // the tile's second half is in the first pair's future where the tile is the workgroup's own
    if (tile < n - 1 || pair) slots<NKS / 2, NKS>([&](auto i) { col_mfma(i); });
  };
  // LDS instructions issued since item i's (or the second's of the two that are waited for together), items up to i + AH - 1 asked for
  auto since = [](int i) constexpr {
    int m = 0;
    for (int y = i == NP ? i + 1 : i + 2; y < i + AH && y <= NP + NKS; ++y) m += y < NP ? 1 : y == NP ? 4 : 2;
    return m;
  };
  auto ask = [&](auto item) __attribute__((always_inline)) {
    constexpr int i = decltype(item)::value;
    if constexpr (i < NP) ask_row(item);
    else if constexpr (i == NP) ask_ds();
    else if constexpr (i <= NP + NKS) ask_col(std::integral_constant<int, i - NP - 1>{});
  };
  auto step = [&](int t) __attribute__((always_inline)) {  // dQ += of tile t, dS of tile t + 1
    begin();
    addresses(t + 1, t);
    slots<0, AH>([&](auto i) { ask(i); });
    start();
    slot_end();
    slots<0, NP + NKS + 1>([&](auto i) {
      constexpr int x = decltype(i)::value;
      if constexpr (x < NP) {
        if constexpr (x % 2 == 0) landed<since(x)>(rf[x], rf[x + 1]);
        row_mfma(i);
      } else if constexpr (x == NP) {
        ds.template landed<since(x)>();
      } else {
        constexpr int c = x - NP - 1;
        if constexpr (c % 2 == 0) landed<since(x)>(cf[c], cf[c + 1]);
        col_mfma(std::integral_constant<int, c>{});
      }
      ask(std::integral_constant<int, x + AH>{});
      if constexpr (x >= 1 && x - 1 < 2 * NL) load_one(t + 3, x - 1);
      // P's words from dP's second MFMA on, dS's from dQ's second on
      constexpr int pf = NKS + 1, df = NP + 2;
      slots<0, 8>([&](auto y) {
        constexpr int w = decltype(y)::value;
        if constexpr (pf + w * NKS / 8 == x) p_word(y);
        if constexpr (df + w * (NKS - 1) / 8 == x) ds_word(y);
      });
      slot_end();
    });
    put(t + 1);
  };

  asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(4 * NL) : "memory");  // tile t0
  rows_of(t0);
#pragma unroll 1
  for (int t = t0; t + 2 < n; ++t) step(t);
  begin();
  if (n - 1 > t0) {
    rows_of(n - 1);
    cols_of(n - 2);
    begin();
  }
  cols_of(n - 1);

  bf16_t* row = dq.p + b * dq.sb + h * dq.sh + (long)myq * dq.st;
  bool stored = false;
  if constexpr (D == 64) {
    if (cs) {  // the rotation needs both halves of the columns: the first wavefront of a pair takes the second's
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
      __syncthreads();   // the stages are free
      f32x4* to = (f32x4*)(lds + pair * 4096) + lane;
      if (half) {
#pragma unroll
        for (int e = 0; e < 4; ++e) to[64 * e] = f32x4{acc[0][4 * e], acc[0][4 * e + 1], acc[0][4 * e + 2], acc[0][4 * e + 3]};
      }
      __syncthreads();
      if (!half) {
        f32x16 both[2];
        both[0] = acc[0];
#pragma unroll
        for (int e = 0; e < 4; ++e) {
          const f32x4 x = to[64 * e];
#pragma unroll
          for (int y = 0; y < 4; ++y) both[1][4 * e + y] = x[y];
        }
        store_grad_row(both, scale, row, cs, sn, myq, lh);
      }
      stored = true;
    }
  }
  if (!stored) {
#pragma unroll
    for (int i = 0; i < MDT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const u32x2 w = {pack2bf(acc[i][4 * j] * scale, acc[i][4 * j + 1] * scale), pack2bf(acc[i][4 * j + 2] * scale, acc[i][4 * j + 3] * scale)};
        *(u32x2*)(row + 32 * (half * MDT + i) + 8 * j + 4 * lh) = w;
      }
  }
  if (half == 0 && lh == 0) {
    stats[(long)bh * T + myq] = myD;
    stats[rows + (long)bh * T + myq] = myL;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into LDS is on its way when it is given back
}

}  // namespace

// cos_t / sin_t: bf16 [T][32] or null, D = 64 only. stats: fp32 [2][B*H][T], written.
int tfb_attn_dq_pair_impl(const void* q, const long* qs, const void* k, const long* ks, const void* v, const long* vs, const void* o,
                          const long* os, const void* go, const long* gos, void* dq, const long* dqs, const float* lse, float* stats, int B, int H,
                          int T, int D, float scale, const void* cos_t, const void* sin_t, int nw, hipStream_t s) {
  const long rows = (long)B * H * T;
  const dim3 grid(T / 64, B * H);
  if (D == 64)
    hipLaunchKernelGGL(attn_dq_pair_kernel<64>, grid, dim3(256), 0, s, mk(q, qs), mk(k, ks), mk(v, vs), mk(go, gos), mk(dq, dqs), stats, rows, T, H,
                       scale, scale * LOG2E, (const bf16_t*)cos_t, (const bf16_t*)sin_t, nw, mk(o, os), lse, first_round(T / 64, B * H, false));
  else
    hipLaunchKernelGGL(attn_dq_pair_kernel<128>, grid, dim3(256), 0, s, mk(q, qs), mk(k, ks), mk(v, vs), mk(go, gos), mk(dq, dqs), stats, rows, T, H,
                       scale, scale * LOG2E, nullptr, nullptr, nw, mk(o, os), lse, first_round(T / 64, B * H, false));
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}
