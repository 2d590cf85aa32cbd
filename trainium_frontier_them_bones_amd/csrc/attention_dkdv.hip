// dK and dV of causal flash attention on gfx950, one block of 128 or 64 keys per workgroup, two wavefronts to every 32 keys: all launches of
// D = 128, and those of D = 64 that do not fill the chip.
//
// The first of a pair ("dV") makes S and P of a 32-query half and dV += dO P, the second ("dK") makes dP and dS of it and dK += Q dS; P
// passes from one to the other through 2 KB of LDS, packed as both hold it, and nothing else does. So a wavefront has one product's
// fragments and one gradient in registers (32 + 64 at D = 128), two of them share each SIMD, and one's MFMAs run under the other's
// vector work and LDS waits. The sums are those of one wavefront doing both in turn, in the same order: the same bits.
// What bounds it: instructions. A 32 x 32 half takes the two 99 + 106 of them at D = 64 (16 MFMAs, 512 cycles) and 134 + 144 at D = 128
// (32, 1024), and a SIMD issues one every 5.7 to 6 cycles from its two wavefronts, as it does from one. So the loop runs over two halves
// whose place in a tile is known (addresses move on once a tile, accumulators alternate without copies).
// One wavefront doing both -> pairs, us: D = 128 (340 registers, alone on its SIMD) B1 H8 T2048 66 -> 52; with dQ's launch B3 H8 T1664
// 109 -> 98, B16 H6 T2048 435 -> 409, B2 H16 T4096 498 -> 466; D = 64 B1 H12 T2048 45 -> 35.6.
// D = 128 has no other kernel: with dQ's launch, over 1 to 512 heads (up to 1536 blocks), pairs take 0.85 - 0.94 of the time at T4096 and T2048,
// 0.89 - 0.97 at T1024 to T512, 0.93 - 1.00 at T384 (96 heads 46.1 -> 46.1), 0.96 - 0.99 at T256 (512 heads 117.8 -> 116.3), and 0.1 - 0.4 us more where a sequence is one
// block (8 heads 22.2 -> 22.4, 256 30.4 -> 30.8, 512 55.5 -> 55.8).
// 64 keys a workgroup (two pairs) where the longest block sets the time: a wavefront alone on its SIMD issues as fast as two together, so half
// the pairs on a CU take half as long (B1 H12 T2048 D64 35.6 -> 28; attention_core.hpp has the line, and both sides of it).
#include "attention_slots.hpp"

namespace {

typedef std::integral_constant<int, 0> H0;
typedef std::integral_constant<int, 1> H1;

struct PBlock {  // a 32 x 32 block of P on its way from one wavefront to another, eight packed words a lane
  u32x4 v[2];
  template <int OFF>
  __device__ __forceinline__ void put(uint32_t at, const uint32_t (&x)[8]) const {
    const u32x4 lo = {x[0], x[1], x[2], x[3]}, hi = {x[4], x[5], x[6], x[7]};
    asm volatile("ds_write_b128 %0, %1 offset:%3\n\tds_write_b128 %0, %2 offset:%4\n\ts_waitcnt lgkmcnt(0)" ::"v"(at), "v"(lo), "v"(hi), "n"(OFF), "n"(OFF + 1024) : "memory");
  }
  template <int OFF>
  __device__ __forceinline__ void get(uint32_t at) {
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v[0]) : "v"(at), "n"(OFF));
    asm volatile("ds_read_b128 %0, %1 offset:%2" : "=v"(v[1]) : "v"(at), "n"(OFF + 1024));
  }
  template <int AFTER>
  __device__ __forceinline__ void landed() {
    asm volatile("s_waitcnt lgkmcnt(%2)" : "+v"(v[0]), "+v"(v[1]) : "n"(AFTER));
  }
};

template <int D, int PAIRS>
__global__ __launch_bounds__(128 * PAIRS, 2) void attn_dkdv_pair_kernel(AttnT q, AttnT k, AttnT v, AttnT go, AttnT dk, AttnT dv,
                                                                const float* __restrict__ stats, long rows, int T, int H, float scale,
                                                                float sl2, const bf16_t* __restrict__ cs, const bf16_t* __restrict__ sn,
                                                                int nw, int turn) {
  typedef Geo<D> G;
  constexpr int TILE = G::TILE, NKS = G::NKS, NDT = G::NDT;
  constexpr int NI = 2 * NKS + 1;            // items of a half: the accumulator's start, NKS row fragments, NKS column fragments
  constexpr int AH = 4;                      // items asked for ahead of their use
  constexpr int KEYS = 32 * PAIRS;
  constexpr int TL = 4 / PAIRS, NL = 16 / G::TPI * TL, SHARE = NL / 2 + 1;  // a wavefront's load instructions for a tile, and for a tile in a half (with statistics)
  constexpr int STAGE = 2 * TILE + 512;      // Q tile, dO tile, 64 x (-lse / scale), 64 x (-delta)
  static_assert(AH <= NKS && 2 * NDT == NKS, "the items ahead of the next half are its start and rows");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[4 * STAGE + 2 * PAIRS * 2048];  // and P: two halves of every pair
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), w = wave % PAIRS;
  int bx, bh;
  xcd_block(T / KEYS, gridDim.y, bx, bh, turn);
  const int b = bh / H, h = bh % H;
  const int nx = T / KEYS, npass = PAIRS == 4 ? paired_passes(nx) : 1;
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void_t*)lds;
  const uint32_t pa = lds0 + 4 * STAGE + w * 2048 + lane * 16;

  // Time goes in steps of one barrier each. In the step that is numbered u by the rows it makes, a dV wavefront does S(u), then dV += of
  // half u - 1 with P(u)'s exponentials between the MFMAs; a dK wavefront dK += of half u - 2 with dS(u - 1) between, then dP(u): the one's
  // bare MFMAs run under the other's vector work. A pair's first half is w, the one on its diagonal. Each role brings the tiles its rows
  // come from: in step u half of tile u / 2 + 2; at the barrier of the odd step 2 i - 1 all of tile i has landed, so that the next
  // step's first fragments may be asked for in front of its barrier.
  auto run = [&](auto ROLE, int pass) __attribute__((always_inline)) {
    constexpr bool DK = decltype(ROLE)::value;
    constexpr int ROWT = DK ? TILE : 0, COLT = DK ? 0 : TILE, STAT = 2 * TILE + (DK ? 256 : 0);
    const int kb = PAIRS == 4 ? paired_block(nx, bx, pass, false) : bx;  // low key blocks see the most query tiles
    const int mykey = kb * KEYS + w * 32 + lr;
    // with a band the keys of a 128-token tile i are seen by the queries of tiles i .. i + nw - 1 only
    const int t0 = kb * (KEYS / 64), nall = T / 64 - t0, nband = 2 * (t0 / 2 + nw) - t0;
    const int nt = nw > 0 && nband < nall ? nband : nall, nh = 2 * nt;  // 64-query tiles, 32-query halves (PAIRS or more)
    const AttnT& rt = DK ? go : q;
    const AttnT& ft = DK ? v : k;
    const long rst = rt.st * 2;
    const uint8_t* rp = (const uint8_t*)(rt.p + b * rt.sb + h * rt.sh + (long)kb * KEYS * rt.st);
    const float* sp = stats + (DK ? 0 : rows) + (long)bh * T + kb * KEYS;
    TileLoad<D, NL / TL> ld[TL];  // (two pairs: each wavefront has two wavefronts' share)
#pragma unroll
    for (int i = 0; i < TL; ++i) ld[i].init(rst, w + 2 * i, lane);
    // (a load past the last tile brings that one again, into a stage nobody reads any more)
    auto load_one = [&](int tile, auto half, int i) __attribute__((always_inline)) {
      constexpr int hf = decltype(half)::value;
      const int from = tile < nt ? tile : nt - 1;
      uint8_t* to = lds + (tile & 3) * STAGE;
      if (i < NL / 2)
        ld[TL == 1 ? 0 : hf].issue_one(TL == 1 ? i + hf * (NL / 2) : i, rp + (long)from * 64 * rst, rst, to + ROWT);
      else
        __builtin_amdgcn_global_load_lds((glb_void_t*)(sp + from * 64 + lane), (lds_void_t*)(to + STAT), 4, 0, 0);
    };
#pragma unroll
    for (int t = 0; t < 2; ++t) {
#pragma unroll
      for (int i = 0; i < SHARE; ++i) load_one(t, H0{}, i);
#pragma unroll
      for (int i = 0; i < SHARE; ++i) load_one(t, H1{}, i);
    }
    bf16x8 ff[NKS];  // K or V of this wavefront's keys
    {
      const bf16_t* fp = ft.p + b * ft.sb + h * ft.sh + (long)mykey * ft.st;
#pragma unroll
      for (int s = 0; s < NKS; ++s) ff[s] = *(const bf16x8*)(fp + 16 * s + 8 * lh);
    }
    f32x16 acc[NDT];
#pragma unroll
    for (int i = 0; i < NDT; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) acc[i][e] = 0.f;

    f32x16 X[2];      // S, or dP, of an even and an odd half
    uint32_t xw[8];   // P, or dS: the columns' operand
    PBlock pb;        // the dK role: P
    RowFrag rf[NKS];
    ColFrag cf[NKS];
    StatFrag sf[2];
    // Addresses of the fragments in the tile that is read: moved on where a tile's first half is asked for, its second is an offset.
    uint32_t ra[NKS], ca[2][NDT], sa;
    auto stage_at = [&](int tile) { return lds0 + (tile & 3) * STAGE; };
    auto set_addresses = [&](int row_tile, int col_tile) __attribute__((always_inline)) {
      FragAddr<D> fr, fc;
      fr.init(stage_at(row_tile), lane);
      fc.init(stage_at(col_tile), lane);
#pragma unroll
      for (int i = 0; i < NKS; ++i) ra[i] = fr.rows[i];
#pragma unroll
      for (int i = 0; i < NDT; ++i) {
        ca[0][i] = fc.lo[i];
        ca[1][i] = fc.hi[i];
      }
      sa = stage_at(row_tile) + 16 * lh;
    };
    auto on = [](int half) { return (uint32_t)((half >> 1) & 3 ? STAGE : -3 * STAGE); };  // to the tile of this half
    auto ask_stat = [&](auto par, uint32_t by) __attribute__((always_inline)) {
      constexpr int p = decltype(par)::value;
      if constexpr (p == 0) sa += by;
      sf[p].template request<STAT + p * 128>(sa);
    };
    auto ask_row = [&](auto item, auto par, uint32_t by) __attribute__((always_inline)) {
      constexpr int i = decltype(item)::value, p = decltype(par)::value;
      if constexpr (p == 0) ra[i] += by;
      rf[i].template request<ROWT + p * (TILE / 2)>(ra[i]);
    };
    auto ask_col = [&](auto item, auto par, uint32_t by) __attribute__((always_inline)) {
      constexpr int i = decltype(item)::value, p = decltype(par)::value, dt = i % NDT;
      if constexpr (p == 0 && i < NDT) {
        ca[0][dt] += by;
        ca[1][dt] += by;
      }
      cf[i].template request<COLT + p * (TILE / 2) + (i / NDT) * 16 * G::ROWB>(ca[0][dt], ca[1][dt]);
    };
    auto use_row = [&](auto item, auto par, auto aft) __attribute__((always_inline)) {
      constexpr int i = decltype(item)::value, p = decltype(par)::value;
      if constexpr (i % 2 == 0) landed<decltype(aft)::value>(rf[i], rf[i + 1]);
      X[p] = mfma_bf16(rf[i].get(), ff[i], X[p]);
    };
    auto use_col = [&](auto item, auto aft) __attribute__((always_inline)) {
      constexpr int i = decltype(item)::value, x = 4 * (i / NDT);
      if constexpr (i % 2 == 0) landed<decltype(aft)::value>(cf[i], cf[i + 1]);
      acc[i % NDT] = mfma_bf16(cf[i].get(), frag_from(xw[x], xw[x + 1], xw[x + 2], xw[x + 3]), acc[i % NDT]);
    };
    auto pair_of = [&](auto word, auto par) __attribute__((always_inline)) {  // two of a lane's sixteen: exponentials, or dS
      constexpr int x = decltype(word)::value, p = decltype(par)::value;
      float a, c;
      if constexpr (DK) {  // the reference multiplies dP - delta by the rounded P
        a = bflo(pb.v[x / 4][x % 4]) * X[p][2 * x];
        c = bfhi(pb.v[x / 4][x % 4]) * X[p][2 * x + 1];
      } else {
        a = X[p][2 * x] * sl2;
        c = X[p][2 * x + 1] * sl2;
        pin(a, c);
        a = fast_exp2(a);
        c = fast_exp2(c);
      }
      pin(a, c);
      X[p][2 * x] = a;
      X[p][2 * x + 1] = c;
    };
    auto word_of = [&](auto word, auto par) __attribute__((always_inline)) {
      constexpr int x = decltype(word)::value, p = decltype(par)::value;
      xw[x] = pack2bf(X[p][2 * x], X[p][2 * x + 1]);
      pin(xw[x]);
    };
    // P's two places alternate
    auto p_put = [&](auto par) __attribute__((always_inline)) { pb.template put<decltype(par)::value * PAIRS * 2048>(pa, xw); };
    auto p_get = [&](auto par) __attribute__((always_inline)) { pb.template get<decltype(par)::value * PAIRS * 2048>(pa); };
    auto begin = [&](auto par) __attribute__((always_inline)) {  // the barrier in front of step u, u > 0
      if constexpr (decltype(par)::value == 1) asm volatile("s_waitcnt vmcnt(%0)" ::"n"(SHARE) : "memory");
      asm volatile("s_barrier" ::: "memory");
    };

    // A step's items in the order of their LDS reads. dV: start and rows of half u, columns of u - 1, and in front of the next barrier
    // the first items of step u + 1. dK: columns of half u - 2, start and rows of u, and the first columns of u - 1.
    auto kind = [](int i) constexpr {  // 0 start, 1 row, 2 column
      const int x = i % NI;
      return DK ? (x < NKS ? 2 : x == NKS ? 0 : 1) : (x == 0 ? 0 : x <= NKS ? 1 : 2);
    };
    auto number = [](int i) constexpr {
      const int x = i % NI;
      return DK ? (x < NKS ? x : x - NKS - 1) : (x <= NKS ? x - 1 : x - NKS - 1);
    };
    auto nlds = [kind](int i) constexpr { return kind(i) == 0 ? 4 : kind(i); };
    auto ask = [&](auto item, auto par, uint32_t byr, uint32_t byc) __attribute__((always_inline)) {  // par: of u
      constexpr int i = decltype(item)::value, p = decltype(par)::value, kd = kind(i), nr = number(i);
      // rows and start: half u, or u + 1 as the dV role's next; columns: u - 1 (dV), u - 2 or as the dK role's next u - 1
      typedef std::integral_constant<int, (kd < 2 ? p + (i >= NI) : DK ? p + (i >= NI) : p + 1) & 1> Par;
      if constexpr (kd == 0) ask_stat(Par{}, byr);
      else if constexpr (kd == 1) ask_row(std::integral_constant<int, nr>{}, Par{}, byr);
      else ask_col(std::integral_constant<int, nr>{}, Par{}, byc);
    };
    auto use = [&](auto item, auto par, auto aft) __attribute__((always_inline)) {
      constexpr int i = decltype(item)::value, kd = kind(i), nr = number(i);
      if constexpr (kd == 0) sf[decltype(par)::value].template landed<decltype(aft)::value>(X[decltype(par)::value]);
      else if constexpr (kd == 1) use_row(std::integral_constant<int, nr>{}, par, aft);
      else use_col(std::integral_constant<int, nr>{}, aft);
    };
    // LDS instructions issued since item i's (or since the second's of the two that are waited for together), when items up to
    // min(i + AH, end) - 1 have been asked for and `extra` other reads behind item AH - 1
    auto since = [kind, number, nlds](int i, int end, int extra) constexpr {
      const int last = kind(i) == 0 ? i : number(i) % 2 == 0 ? i + 1 : i;
      int n = last < AH ? extra : 0;
      for (int y = last + 1; y < i + AH && y < end; ++y) n += nlds(y);
      return n;
    };
    constexpr int CP = NKS == 8 ? 2 : 1;  // the dK role: the column slot behind which P is there
    // a full step; par: of u
    auto step = [&](int u, auto par) __attribute__((always_inline)) {
      constexpr int p = decltype(par)::value;
      typedef std::integral_constant<int, 1 - p> Other;
      typedef std::integral_constant<int, DK ? 1 - p : p> Elem;  // whose exponentials or dS
      begin(par);
      // (only one of a step's two kinds of address moves on at its parity)
      const uint32_t byr = DK || p == 0 ? on(u) : on(u + 1), byc = DK ? (p == 0 ? on(u - 2) : on(u - 1)) : on(u - 1);
      if constexpr (DK) p_get(Other{});
      const int tile = (u >> 1) + 2;
      slot_end();
      slots<0, NI>([&](auto i) {
        constexpr int x = decltype(i)::value;
        use(i, par, std::integral_constant<int, since(x, 1 << 20, DK ? 2 : 0)>{});
        constexpr int c = kind(x) == 2 ? number(x) : -1;
        if constexpr (DK && c == CP) {
          constexpr auto n = [nlds]() constexpr {
            int m = 0;
            for (int y = AH; y < AH + CP; ++y) m += nlds(y);
            return m;
          };
          pb.template landed<n()>();
        }
        ask(std::integral_constant<int, x + AH>{}, par, byr, byc);
        if constexpr (x % 2 == 1 && x / 2 < SHARE) load_one(tile, par, x / 2);
        constexpr int first = CP;
        if constexpr (c >= first)
          slots<0, 8>([&](auto y) { if constexpr (first + decltype(y)::value * (NKS - first) / 8 == c) pair_of(y, Elem{}); });
        if constexpr (c >= NKS / 2)
          slots<0, 4>([&](auto y) { if constexpr (NKS / 2 + decltype(y)::value * NKS / 8 == c) word_of(y, Elem{}); });
        if constexpr (c == NKS - 1) slots<4, 8>([&](auto y) { word_of(y, Elem{}); });
        slot_end();
      });
      if constexpr (!DK) p_put(par);
    };

    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(2 * SHARE) : "memory");  // tile 0
    auto begin_at = [&](int u) __attribute__((always_inline)) {
      if (u & 1) begin(H1{});
      else if (u > 0) begin(H0{});
    };
    auto load_share = [&](int u) __attribute__((always_inline)) {
      if (u & 1) {
#pragma unroll
        for (int i = 0; i < SHARE; ++i) load_one((u >> 1) + 2, H1{}, i);
      } else {
#pragma unroll
        for (int i = 0; i < SHARE; ++i) load_one((u >> 1) + 2, H0{}, i);
      }
    };
    // The parts of a step by themselves, in front of the loop and behind it. Nothing is left in flight: where ways of the program meet,
    // registers are copied.
    constexpr int XI = DK ? 1 : 0;
    typedef std::integral_constant<int, XI> Xi;
    auto rows_of = [&](int u) __attribute__((always_inline)) {
      FragAddr<D> f;
      f.init(stage_at(u >> 1) + (u & 1) * (TILE / 2), opaque(lane));
      sf[XI].template request<STAT>(stage_at(u >> 1) + (u & 1) * 128 + 16 * opaque(lh));
      slots<0, NKS>([&](auto i) { rf[decltype(i)::value].template request<ROWT>(f.rows[decltype(i)::value]); });
      sf[XI].template landed<0>(X[XI]);
      slots<0, NKS>([&](auto i) { use_row(i, Xi{}, std::integral_constant<int, 0>{}); });
    };
    auto cols_of = [&](int u) __attribute__((always_inline)) {
      FragAddr<D> f;
      f.init(stage_at(u >> 1) + (u & 1) * (TILE / 2), opaque(lane));
      slots<0, 2>([&](auto ks) {
        constexpr int c0 = decltype(ks)::value * NDT;
        slots<0, NDT>([&](auto i) {
          constexpr int dt = decltype(i)::value;
          cf[c0 + dt].template request<COLT + (c0 / NDT) * 16 * G::ROWB>(f.lo[dt], f.hi[dt]);
        });
        slots<c0, c0 + NDT>([&](auto i) { use_col(i, std::integral_constant<int, 0>{}); });
      });
    };
    auto elem_of = [&]() __attribute__((always_inline)) {
      slots<0, 8>([&](auto i) {
        pair_of(i, Xi{});
        word_of(i, Xi{});
      });
    };
    auto p_put_at = [&](int u) __attribute__((always_inline)) { pb.template put<0>(pa + (u & 1) * (PAIRS * 2048), xw); };
    auto p_get_at = [&](int u) __attribute__((always_inline)) {
      pb.template get<0>(pa + (u & 1) * (PAIRS * 2048));
      pb.template landed<0>();
    };

    for (int u = 0; u < w; ++u) {  // steps in front of this pair's first
      begin_at(u);
      load_share(u);
    }
    begin_at(w);
    load_share(w);
    rows_of(w);
    // up to an even step; the loop (nh is even)
    const int u0 = DK ? (w + 3) & ~1 : (w + 2) & ~1;
    if constexpr (!DK) {
      const int kq = lr - 4 * lh;  // key - q for element e is kq - (e>>2)*8 - (e&3)
#pragma unroll
      for (int e = 0; e < 16; ++e) X[0][e] = (kq - 8 * (e >> 2) - (e & 3) > 0) ? -INFINITY : X[0][e];
      elem_of();
      p_put_at(w);
    }
#pragma unroll 1
    for (int u = w + 1; u < u0 && u < nh; ++u) {
      begin_at(u);
      load_share(u);
      if constexpr (DK) {
        p_get_at(u - 1);
        if (u > w + 1) cols_of(u - 2);
        elem_of();
        rows_of(u);
      } else {
        rows_of(u);
        cols_of(u - 1);
        elem_of();
        p_put_at(u);
      }
    }
    set_addresses((u0 >> 1) - 1, (u0 >> 1) - (DK ? 2 : 1));
    if (u0 < nh) {
      slots<0, AH>([&](auto i) { ask(i, H0{}, on(u0), on(u0 - 2)); });
#pragma unroll 1
      for (int u = u0; u < nh; u += 2) {
        step(u, H0{});
        step(u + 1, H1{});
      }
      // (the items asked for are not used, but their registers are theirs until they have landed)
      if constexpr (DK) {
        slots<0, AH>([&](auto i) { if constexpr (decltype(i)::value % 2 == 0) landed<0>(cf[decltype(i)::value], cf[decltype(i)::value + 1]); });
      } else {
        sf[0].template landed<0>(X[0]);
        slots<0, AH - 1>([&](auto i) { pin(rf[decltype(i)::value].v); });
      }
    }
    begin(H0{});
    if constexpr (DK) {
      p_get_at(nh - 1);
      if (nh - 2 >= w) cols_of(nh - 2);
      elem_of();
    }
    cols_of(nh - 1);
    const AttnT& gt = DK ? dk : dv;
    bf16_t* row = gt.p + b * gt.sb + h * gt.sh + (long)mykey * gt.st;
    if constexpr (D == 64) store_grad_row(acc, DK ? scale : 1.0f, row, DK ? cs : nullptr, DK ? sn : nullptr, mykey, lh);
    else store_grad_row<D>(acc, DK ? scale : 1.0f, row, lh);
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  };
  for (int pass = 0; pass < npass; ++pass) {
    if (wave < PAIRS) run(std::false_type{}, pass);
    else run(std::true_type{}, pass);
    if (pass + 1 < npass) __syncthreads();  // the stages are free for the partner block
  }
}

}  // namespace

// stats: fp32 [2][B*H][T] (-delta, then -lse / scale), as the dQ kernels leave them. cos_t / sin_t: bf16 [T][32] or null, D = 64 only.
int tfb_attn_dkdv_impl(const void* q, const long* qs, const void* k, const long* ks, const void* v, const long* vs, const void* go,
                       const long* gos, void* dk, const long* dks, void* dv, const long* dvs, const float* stats, int B, int H, int T,
                       int D, float scale, const void* cos_t, const void* sin_t, int nw, hipStream_t s) {
  const long rows = (long)B * H * T, nbh = (long)B * H;
  const bool half = tfb_attn_dkdv_half_applies(D, T, nbh, nw, qs, gos);
  const dim3 grid(half ? T / 64 : paired_grid(T / 128, B * H, 1), B * H), block(half ? 256 : 512);
  const bf16_t *cs = D == 64 ? (const bf16_t*)cos_t : nullptr, *sn = D == 64 ? (const bf16_t*)sin_t : nullptr;
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, block, 0, s, mk(q, qs), mk(k, ks), mk(v, vs), mk(go, gos), mk(dk, dks), mk(dv, dvs), stats, rows, T, H, scale,
                       scale * LOG2E, cs, sn, nw, half ? first_round(T / 64, B * H, false) : 0);
  };
  if (D == 64) half ? launch(attn_dkdv_pair_kernel<64, 2>) : launch(attn_dkdv_pair_kernel<64, 4>);
  else half ? launch(attn_dkdv_pair_kernel<128, 2>) : launch(attn_dkdv_pair_kernel<128, 4>);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}
