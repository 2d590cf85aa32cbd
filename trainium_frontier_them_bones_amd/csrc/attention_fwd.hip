// Causal flash attention forward on gfx950 for launches that do not fill the chip: 64 queries per workgroup, two wavefronts to every 32.
//
// With one wavefront to 32 queries the longest block sets such a launch's time, and a wavefront alone on its SIMD takes all of its
// instructions in turn. Here the first of a pair ("P") makes the scores, the row maximum and P of a 64-key tile and hands P to the other
// through 4 KB of LDS; the second ("O") adds P V and the row sum of the tile before and brings the tiles. A row's reference point is P's
// alone: where it moves, its factor goes along with the tile. The sums are those of one wavefront doing both in turn, in the same order: the
// same bits.
// What bounds it: P's instructions, some 140 a tile at D = 64 with 32 exponentials and 8 MFMAs among them (O has half as many, and the loads). With
// the keys of a tile divided between the two, P and the row maximum passed both ways, it takes as long (B1 H12 T2048 D64 23.1 us, this 22.4);
// with a row maximum and sums of its own for each half less (19.9), but with other bits than a larger batch. K's first fragments asked for a
// barrier early, or two of the loads made by P: 22.6, 24.2. us, one wavefront to 32 queries -> this: B1 H12 T2048 D64 25.7 -> 22.4, B1 H8 T2048 D128
// 31.9 -> 29.9; attention_core.hpp has the line.
#include "attention_slots.hpp"

namespace {

struct PTile {  // P of 32 queries and 64 keys, packed: fragment i is the operand of the 16 keys i
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
__global__ __launch_bounds__(256, 2) void attn_fwd_pair_kernel(AttnT q, AttnT k, AttnT v, AttnT o, float* __restrict__ lse, int T, int H, float sl2,
                                                               int nw, int turn) {
  typedef Geo<D> G;
  constexpr int TILE = G::TILE, NKS = G::NKS, NDT = G::NDT, NA = 2 * NKS, NO = 4 * NDT;  // score MFMAs of a tile, output MFMAs
  constexpr int AH = 4;                          // fragments asked for ahead of their MFMA
  constexpr int NL = 16 / G::TPI;                // a quarter of a K or V tile's load instructions
  constexpr int NBK = 4, NBV = 3, WPS = 16 / NA; // LDS buffers for K tiles and for V tiles; packed pairs of scores to a slot
  // behind the tiles, for two tiles in turn: P of two pairs, the factors (then the last reference points), whether they are wanted
  constexpr int PX = (NBK + NBV) * TILE, AX = PX + 2 * 8192, FX = AX + 3 * 512;
  static_assert(NO == NA && 16 % NA == 0, "slots");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[FX + 64];
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6), pair = wave >> 1;
  const int nx = T / 64;
  int bx, bh;
  xcd_block(nx, gridDim.y, bx, bh, turn);
  const int b = bh / H, h = bh % H, qb = nx - 1 - bx;   // the most tiles first
  const int myq = qb * 64 + pair * 32 + lr;
  const int n = qb + 1, t0 = band_first_tile(qb >> 1, nw);  // tile n - 1 is over the workgroup's own tokens
  const uint32_t lds0 = (uint32_t)(uintptr_t)(lds_void_t*)lds;
  const uint32_t pa = lds0 + PX + pair * 4096 + lane * 16, xa = lds0 + AX + pair * 256 + lane * 4, ga = lds0 + FX + pair * 4;
  FragAddr<D> fa;
  fa.init(lds0, lane);
  auto next_k = [](int buf) { return buf == NBK - 1 ? 0 : buf + 1; };
  auto next_v = [](int buf) { return buf == NBV - 1 ? 0 : buf + 1; };
  constexpr std::integral_constant<int, 0> even{};
  constexpr std::integral_constant<int, 1> odd{};
  // Time goes in steps of one barrier each, t0 .. n: in step t a P wavefront makes P of tile t and the scores of tile t + 1, an O wavefront
  // adds tile t - 1.
  if ((wave & 1) == 0) {
    bf16x8 qf[NKS];
    {
      const bf16_t* qr = q.p + b * q.sb + h * q.sh + (long)myq * q.st;
#pragma unroll
      for (int s = 0; s < NKS; ++s) qf[s] = *(const bf16x8*)(qr + 16 * s + 8 * lh);
    }
    f32x16 scA[2], scB[2];  // raw scores S = K Q^T of an even and an odd tile (key = MFMA row: a lane holds 32 keys of one query)
    uint32_t pw[16];
    RowFrag kf[NA];
    uint32_t ka[NKS];
    float m = -1e30f, mx = 0.f, mx1 = 0.f, alpha = 1.f;  // running maximum of the raw scores
    int grow = 0;
    typedef std::integral_constant<int, 0> C0;
    auto k_at = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int s = 0; s < NKS; ++s) ka[s] = fa.rows[s] + buf * TILE;
    };
    auto request = [&](auto item) __attribute__((always_inline)) {
      constexpr int i = decltype(item)::value;
      if constexpr (i < NA) kf[i].template request<(i / NKS) * 32 * G::ROWB>(ka[i % NKS]);
    };
    auto score_slot = [&](auto slot, f32x16 (&sn)[2]) __attribute__((always_inline)) {
      constexpr int i = decltype(slot)::value, kt = i / NKS, s = i % NKS;
      if constexpr (i % 2 == 0) landed<(i + AH <= NA ? AH - 2 : NA - 2 - i)>(kf[i], kf[i + 1]);
      if constexpr (s == 0) sn[kt] = mfma_bf16(kf[i].get(), qf[s], f32x16{});
      else sn[kt] = mfma_bf16(kf[i].get(), qf[s], sn[kt]);
      request(std::integral_constant<int, i + AH>{});
    };
    // P = exp2(sl2 (S - m)) rounded to bf16, WPS words (two scores each) at a time
    auto exp_words = [&](auto w, const f32x16 (&sc)[2], float negm) __attribute__((always_inline)) {
      constexpr int w0 = decltype(w)::value, kt = w0 >> 3, e0 = 2 * (w0 & 7);
      float f[2 * WPS];
#pragma unroll
      for (int e = 0; e < 2 * WPS; ++e) f[e] = fmaf(sc[kt][e0 + e], sl2, negm);
#pragma unroll
      for (int e = 0; e < 2 * WPS; ++e) f[e] = fast_exp2(f[e]);
#pragma unroll
      for (int e = 0; e < WPS; ++e) {
        pw[w0 + e] = pack2bf(f[2 * e], f[2 * e + 1]);
        pin(pw[w0 + e]);
      }
    };
    auto put_word = [](uint32_t at, float x) __attribute__((always_inline)) { asm volatile("ds_write_b32 %0, %1" ::"v"(at), "v"(x) : "memory"); };
    auto put_p = [&](auto par) __attribute__((always_inline)) {
      constexpr int P = decltype(par)::value;
      const u32x4 w0 = {pw[0], pw[1], pw[2], pw[3]}, w1 = {pw[4], pw[5], pw[6], pw[7]}, w2 = {pw[8], pw[9], pw[10], pw[11]},
                  w3 = {pw[12], pw[13], pw[14], pw[15]};
      const uint32_t at = pa + P * 8192;
      asm volatile("ds_write_b128 %0, %1\n\tds_write_b128 %0, %2 offset:1024\n\tds_write_b128 %0, %3 offset:2048\n\tds_write_b128 %0, %4 offset:3072" ::"v"(at),
                   "v"(w0), "v"(w1), "v"(w2), "v"(w3) : "memory");
      put_word(ga + P * 8, __builtin_bit_cast(float, grow));
      if (grow) put_word(xa + P * 512, alpha);
    };
    // the row maximum with a tile's scores. The reference point of the exponentials follows it only when some row's has grown by more than
    // 2^8: O and lse do not depend on it.
    auto max_first = [&](auto from, auto to, const f32x16 (&sc)[2]) __attribute__((always_inline)) {  // of the tile's first half
#pragma unroll
      for (int i = decltype(from)::value; i < decltype(to)::value; ++i) mx = fmaxf(fmaxf(mx, sc[0][2 * i]), sc[0][2 * i + 1]);
    };
    auto follow = [&](int tile, f32x16 (&sc)[2]) __attribute__((always_inline)) {  // behind max_first
      if (tile == n - 1) {  // over the workgroup's own tokens
        const int kbase = opaque(lh * 4 - pair * 32 - lr);  // key - q of element (kt, e) is kbase + 32 kt + (e >> 2) * 8 + (e & 3)
#pragma unroll
        for (int kt = 0; kt < 2; ++kt)
#pragma unroll
          for (int e = 0; e < 16; ++e) sc[kt][e] = (kbase + kt * 32 + (e >> 2) * 8 + (e & 3) > 0) ? -INFINITY : sc[kt][e];
        mx = m;
        max_first(C0{}, std::integral_constant<int, 8>{}, sc);
      }
      mx1 = m;
#pragma unroll
      for (int e = 0; e < 16; e += 4) {  // (two chains)
        mx1 = fmaxf(fmaxf(mx1, sc[1][e]), sc[1][e + 1]);
        mx = fmaxf(fmaxf(mx, sc[1][e + 2]), sc[1][e + 3]);
      }
      mx = max_halves(fmaxf(mx, mx1));
      grow = __builtin_amdgcn_ballot_w64((mx - m) * sl2 > 8.0f) != 0;
      if (grow) {
        alpha = fast_exp2((m - mx) * sl2);
        m = mx;
      }
    };
    auto begin = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); };
    int kb = 0;  // the buffer of K t + 1
    // the next tile's first fragments, asked for in front of the barrier
    auto ask_next = [&]() __attribute__((always_inline)) {
      kb = next_k(kb);
      k_at(kb);
      slots<0, AH>([&](auto i) { request(i); });
    };
    auto have_next = [&]() __attribute__((always_inline)) {
      begin();
      landed<0>(kf[0], kf[1]);
      landed<0>(kf[2], kf[3]);
    };
    // step t, behind its barrier
    auto step = [&](auto par, int t, const f32x16 (&sc)[2], f32x16 (&sn)[2]) __attribute__((always_inline)) {
      const float negm = -m * sl2;
      mx = m;
      slot_end();
      slots<0, NA>([&](auto i) {
        constexpr int x = decltype(i)::value;
        score_slot(i, sn);
        exp_words(std::integral_constant<int, x * WPS>{}, sc, negm);
        if constexpr (x >= NA - 2) max_first(std::integral_constant<int, x == NA - 2 ? 0 : 4>{}, std::integral_constant<int, x == NA - 2 ? 4 : 8>{}, sn);
        slot_end();
      });
      put_p(par);
      ask_next();
      slot_end();
      follow(t + 1, sn);
      have_next();
    };
    auto last_step = [&](auto par, const f32x16 (&sc)[2]) __attribute__((always_inline)) {
      const float negm = -m * sl2;
      slots<0, NA>([&](auto i) { exp_words(std::integral_constant<int, decltype(i)::value * WPS>{}, sc, negm); });
      put_p(par);
      put_word(xa + 2 * 512, m);
      begin();
    };
    asm volatile("s_barrier" ::: "memory");  // K of tiles t0 and t0 + 1
    k_at(0);
    slots<0, AH>([&](auto i) { request(i); });
    slots<0, NA>([&](auto i) { score_slot(i, scA); });
    ask_next();
    mx = m;
    max_first(C0{}, std::integral_constant<int, 8>{}, scA);
    follow(t0, scA);
    have_next();
    int t = t0;
#pragma unroll 1
    for (; t + 2 < n; t += 2) {
      step(even, t, scA, scB);
      step(odd, t + 1, scB, scA);
    }
    if (t + 1 < n) {
      step(even, t, scA, scB);
      last_step(odd, scB);
    } else {
      last_step(even, scA);
    }
  } else {
    const long kst = k.st * 2, vst = v.st * 2;
    const uint8_t* kp = (const uint8_t*)(k.p + b * k.sb + h * k.sh);
    const uint8_t* vp = (const uint8_t*)(v.p + b * v.sb + h * v.sh);
    TileLoad<D, NL> lk[2], lv[2];  // (each brings half of a tile: the shares of two of four wavefronts)
#pragma unroll
    for (int x = 0; x < 2; ++x) {
      lk[x].init(kst, pair + 2 * x, lane);
      lv[x].init(vst, pair + 2 * x, lane);
    }
    // (a load past the last tile brings that one again, into a buffer that no result comes from any more)
    auto load_k = [&](int t, int buf, int i) __attribute__((always_inline)) {
      lk[i / NL].issue_one(i % NL, kp + (long)(t < n ? t : n - 1) * 64 * kst, kst, lds + buf * TILE);
    };
    auto load_v = [&](int t, int buf, int i) __attribute__((always_inline)) {
      lv[i / NL].issue_one(i % NL, vp + (long)(t < n ? t : n - 1) * 64 * vst, vst, lds + (NBK + buf) * TILE);
    };
#pragma unroll
    for (int t = 0; t < 4; ++t)
#pragma unroll
      for (int i = 0; i < 2 * NL; ++i) load_k(t0 + t, t, i);
#pragma unroll
    for (int i = 0; i < 2 * NL; ++i) load_v(t0, 0, i);

    f32x16 oacc[NDT];
    float l = 0.f;
#pragma unroll
    for (int i = 0; i < NDT; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) oacc[i][e] = 0.f;
    PTile pt;
    ColFrag vf[NO];
    uint32_t la[NDT], ha[NDT];
    auto v_at = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
      for (int i = 0; i < NDT; ++i) {
        la[i] = fa.lo[i] + (NBK + buf) * TILE;
        ha[i] = fa.hi[i] + (NBK + buf) * TILE;
      }
    };
    auto request = [&](auto item) __attribute__((always_inline)) {
      constexpr int i = decltype(item)::value;
      if constexpr (i < NO) vf[i].template request<(i / NDT) * 16 * G::ROWB>(la[i % NDT], ha[i % NDT]);
    };
    // In front of step t: K of tiles t + 1 and t + 2 and V of tile t - 1 have landed, P of tile t - 1 is in LDS; the buffers of K t and V t - 2 are free.
    auto begin = [&]() __attribute__((always_inline)) { asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(4 * NL) : "memory"); };
    int kb = 0, vb = 0;  // the buffers that step t fills: K t + 4; and reads: V t - 1 (it fills V t + 1)
    auto get_word = [](uint32_t at) __attribute__((always_inline)) {
      float x;
      asm volatile("ds_read_b32 %0, %1" : "=v"(x) : "v"(at));
      return x;
    };
    auto add_tile = [&](auto par, int t, auto more) __attribute__((always_inline)) {  // step t: tile t - 1 (par: its parity from t0)
      constexpr int P = decltype(par)::value;
      float flag = get_word(ga + P * 8);
      pt.request(pa + P * 8192);
      v_at(vb);
      slots<0, AH>([&](auto i) { request(i); });
      const int kfill = kb, vfill = next_v(next_v(vb));
      asm volatile("s_waitcnt lgkmcnt(%1)" : "+v"(flag) : "n"(4 + 2 * AH));
      if (__builtin_amdgcn_readfirstlane(__builtin_bit_cast(int, flag))) {
        float alpha = get_word(xa + P * 512);
        asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(alpha));
        l *= alpha;
#pragma unroll
        for (int i = 0; i < NDT; ++i)
#pragma unroll
          for (int e = 0; e < 16; ++e) oacc[i][e] *= alpha;
      }
      pt.template landed<2 * AH>();
      slot_end();
      slots<0, NO>([&](auto slot) {
        constexpr int i = decltype(slot)::value;
        if constexpr (i % 2 == 0) landed<2 * (i + AH <= NO ? AH - 2 : NO - 2 - i)>(vf[i], vf[i + 1]);
        oacc[i % NDT] = mfma_bf16(vf[i].get(), __builtin_bit_cast(bf16x8, pt.v[i / NDT]), oacc[i % NDT]);
        request(std::integral_constant<int, i + AH>{});
        if constexpr (decltype(more)::value && i < 4 * NL) {
          if constexpr (i < 2 * NL) load_k(t + 4, kfill, i);
          else load_v(t + 1, vfill, i - 2 * NL);
        }
        // the row sum runs over the rounded values
#pragma unroll
        for (int w = i * 16 / NO; w < (i + 1) * 16 / NO; ++w) l = sum2bf(pt.v[w / 4][w % 4], l);
        pin(l);
        slot_end();
      });
      kb = next_k(kb);
      vb = next_v(vb);
    };
    constexpr std::true_type yes{};
    constexpr std::false_type no{};
    asm volatile("s_waitcnt vmcnt(%0)\n\ts_barrier" ::"n"(6 * NL) : "memory");  // K of tiles t0 and t0 + 1
    begin();                                                                    // step t0: nothing to add yet
#pragma unroll
    for (int i = 0; i < 2 * NL; ++i) load_k(t0 + 4, 0, i);
#pragma unroll
    for (int i = 0; i < 2 * NL; ++i) load_v(t0 + 1, 1, i);
    kb = 1;
    int t = t0 + 1;
#pragma unroll 1
    for (; t + 1 < n; t += 2) {
      begin();
      add_tile(even, t, yes);
      begin();
      add_tile(odd, t + 1, yes);
    }
    bool is_odd = false;  // of the last tile
    if (t < n) {
      begin();
      add_tile(even, t, yes);
      ++t;
      is_odd = true;
    }
    begin();  // step n
    if (is_odd) add_tile(odd, t, no);
    else add_tile(even, t, no);
    float m = get_word(xa + 2 * 512);
    asm volatile("s_waitcnt lgkmcnt(0)" : "+v"(m));
    l += __shfl_xor(l, 32, 64);
    const float inv = 1.0f / l;
    bf16_t* orow = o.p + b * o.sb + h * o.sh + (long)myq * o.st;
#pragma unroll
    for (int i = 0; i < NDT; ++i)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const u32x2 w = {pack2bf(oacc[i][4 * j] * inv, oacc[i][4 * j + 1] * inv), pack2bf(oacc[i][4 * j + 2] * inv, oacc[i][4 * j + 3] * inv)};
        *(u32x2*)(orow + 32 * i + 8 * j + 4 * lh) = w;
      }
    if (lh == 0) lse[(long)bh * T + myq] = (m * sl2 + log2f(l)) * LN2;  // m is the raw-score maximum
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into LDS is on its way when it is given back
  }
}

}  // namespace

int tfb_attn_fwd_pair_impl(const void* q, const long* qs, const void* k, const long* ks, const void* v, const long* vs, void* o, const long* os,
                           float* lse, int B, int H, int T, int D, float scale, int nw, hipStream_t s) {
  const dim3 grid(T / 64, B * H);
  const auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid, dim3(256), 0, s, mk(q, qs), mk(k, ks), mk(v, vs), mk(o, os), lse, T, H, scale * LOG2E, nw, first_round(T / 64, B * H, false));
  };
  if (D == 64) launch(attn_fwd_pair_kernel<64>);
  else launch(attn_fwd_pair_kernel<128>);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}
