// Causal flash attention for head dimension 128 on gfx950 (the reference's own models run D = 128): the kernels the C-ABI
// entry points in attention.hip run for D = 128. Same arithmetic contract as the other head dimension (stated in
// attention.hip) and the same data movement as the D = 64 kernels:
//   * 64-token x D tiles go from global memory straight into LDS with global_load_lds_dwordx4 (no staging registers, no
//     VALU transposes); a token's row is 2 D bytes and 16-byte chunk c of token t sits at slot c ^ swz(t), a swizzle under
//     which ONE copy of a tile serves both MFMA operand forms without bank conflicts: token-major fragments (ds_read_b128:
//     16 consecutive tokens of one chunk on 16 different 16-byte bank groups) and transposed fragments
//     (ds_read_b64_tr_b16: the four tokens of a 32-lane access on four different 64-byte bank quarters);
//   * two to four LDS stages, one barrier per stage, the next stages' loads in flight behind it;
//   * workgroups re-dealt so that all sequence blocks of a (batch, head) pair run on one XCD (its L2 then serves the K/V or
//     Q/dO tiles those blocks stream repeatedly), and a workgroup does block i and then block nx - 1 - i (equal causal work
//     per workgroup);
//   * a wavefront owns 32 queries (forward, dQ) or 32 keys (dK/dV) as the MFMA column index: row statistics are per-lane
//     scalars and the packed score registers are directly the B operand of the second product;
//   * the backward accumulators start from the rows' -lse / scale and -delta, which the dQ kernel makes from the dO
//     fragments it holds anyway and leaves for dK/dV.
// The tile loops are software-pipelined by hand, slot by slot: an MFMA, the LDS read of a fragment that a later slot uses, and a
// share of the elementwise work of the neighbouring tile. What bounds them: two wavefronts per SIMD (forward, dQ: all 256 registers)
// share the matrix pipe, which an MFMA holds for 32 cycles and a dot product (the rounded row sum) for about 16; one wavefront alone
// on its SIMD (when the grid leaves CUs half empty) issues an instruction every five cycles, so there the count of instructions per MFMA
// is the time. dK/dV runs in pairs of wavefronts (attention_dkdv.hip).
// Before, with plain loops whose LDS reads stood right in front of their MFMAs -> now: B3 H8 T1664 forward 52 -> 35 us; B1 H8 T2048
// 56 -> 35; B16 H6 T2048 155 -> 120.
#include "attention_slots.hpp"

namespace {

// =========================================================================================== forward
template <int D>
__global__ __launch_bounds__(256, 2) void attnD_fwd_kernel(AttnT q, AttnT k, AttnT v, AttnT o, float* __restrict__ lse, int T,
                                                           int H, float sl2, int nw, int turn) {
  typedef Geo<D> G;
  constexpr int TILE = G::TILE, NKS = G::NKS, NDT = G::NDT, NA = 2 * NKS, NB = 4 * NDT;
  constexpr int AH = 4;  // fragments asked for ahead of their MFMA (6: no register left, 1 % slower)
  static_assert(NA == 16 && NB == 16, "a slot for each packed pair of scores");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[4 * TILE];  // K even, K odd, V even, V odd tile
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int bx, bh;
  xcd_block(T / 128, gridDim.y, bx, bh, turn);
  const int b = bh / H, h = bh % H;
  const bf16_t* qp = q.p + b * q.sb + h * q.sh;
  const uint8_t* kp = (const uint8_t*)(k.p + b * k.sb + h * k.sh);
  const uint8_t* vp = (const uint8_t*)(v.p + b * v.sb + h * v.sh);
  bf16_t* op = o.p + b * o.sb + h * o.sh;
  const int nx = T / 128, npass = paired_passes(nx);
  const long kst = k.st * 2, vst = v.st * 2;
  TileLoad<D, 16 / G::TPI> lk, lv;
  lk.init(kst, wave, lane);
  lv.init(vst, wave, lane);
  auto issue_k = [&](int tile) { lk.issue(kp + (long)tile * 64 * kst, kst, lds + (tile & 1) * TILE); };
  auto issue_v = [&](int tile) { lv.issue(vp + (long)tile * 64 * vst, vst, lds + (2 + (tile & 1)) * TILE); };
  FragAddr<D> fa;
  fa.init((uint32_t)(uintptr_t)(lds_void_t*)lds, lane);

  for (int pass = 0; pass < npass; ++pass) {
    const int qb = paired_block(nx, bx, pass, true);
    const int q0 = qb * 128, qw0 = q0 + wave * 32;
    bf16x8 qf[NKS];
#pragma unroll
    for (int s = 0; s < NKS; ++s) qf[s] = *(const bf16x8*)(qp + (long)(qw0 + lr) * q.st + 16 * s + 8 * lh);
    const int n = (q0 + 128) / 64;               // even; tiles n - 2 and n - 1 cover the workgroup's own 128 tokens
    const int t0 = band_first_tile(qb, nw);      // even
    const int last = n - 2 + (wave >> 1);        // the wavefront's diagonal tile; tiles beyond are in its future
    issue_k(t0);
    issue_v(t0);
    issue_k(t0 + 1);

    f32x16 oacc[NDT];
    float m = -1e30f, l = 0.f;  // running maximum of the raw scores, running sum
#pragma unroll
    for (int i = 0; i < NDT; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) oacc[i][e] = 0.f;
    f32x16 scA[2], scB[2];  // raw scores S = K Q^T of an even and an odd tile (key = MFMA row: a lane holds 32 keys of one query)
    uint32_t pA[16], pB[16];
    RowFrag kf[NA];
    ColFrag vf[NB];
    float mx = 0.f, mx1 = 0.f;  // (two chains)

    auto request = [&](auto par, auto slot) {  // slots 0 .. NA - 1: K of the next tile, then V of this one; par: this tile's parity
      constexpr int i = decltype(slot)::value, P = decltype(par)::value;
      if constexpr (i < NA) kf[i].template request<(P ^ 1) * TILE + (i / NKS) * 32 * G::ROWB>(fa.rows[i % NKS]);
      else if constexpr (i < NA + NB)
        vf[i - NA].template request<(2 + P) * TILE + ((i - NA) / NDT) * 16 * G::ROWB>(fa.lo[(i - NA) % NDT], fa.hi[(i - NA) % NDT]);
    };
    auto score_slot = [&](auto slot, f32x16 (&sn)[2]) {
      constexpr int i = decltype(slot)::value, kt = i / NKS, s = i % NKS;
      constexpr int after = i + AH <= NA ? AH - 2 : (NA - 2 - i) + 2 * (i + AH - NA);
      if constexpr (i % 2 == 0) landed<after>(kf[i], kf[i + 1]);
      const bf16x8 f = kf[i].get();
      if constexpr (s == 0) sn[kt] = mfma_bf16(f, qf[s], f32x16{});
      else sn[kt] = mfma_bf16(f, qf[s], sn[kt]);
    };
    auto out_slot = [&](auto slot, const uint32_t (&pw)[16]) {
      constexpr int i = decltype(slot)::value;
      constexpr int after = 2 * (i + AH <= NB ? AH - 2 : NB - 2 - i);
      if constexpr (i % 2 == 0) landed<after>(vf[i], vf[i + 1]);
      const bf16x8 f = vf[i].get();
      constexpr int g = i / NDT;
      oacc[i % NDT] = mfma_bf16(f, frag_from(pw[4 * g], pw[4 * g + 1], pw[4 * g + 2], pw[4 * g + 3]), oacc[i % NDT]);
    };
    // P = exp2(sl2 (S - m)) rounded to bf16, word by word (two scores), a word's steps in different slots so that none waits for the
    // one before; the row sum runs over the rounded values
    float f0, f1;
    auto step_f = [&](auto word, const f32x16 (&sc)[2], float negm) {
      constexpr int i = decltype(word)::value, kt = i >> 3, e = 2 * (i & 7);
      f0 = fmaf(sc[kt][e], sl2, negm);
      f1 = fmaf(sc[kt][e + 1], sl2, negm);
      pin(f0, f1);
    };
    auto step_x = [&]() {
      f0 = fast_exp2(f0);
      f1 = fast_exp2(f1);
      pin(f0, f1);
    };
    auto step_c = [&](auto word, uint32_t (&pw)[16]) {
      pw[decltype(word)::value] = pack2bf(f0, f1);
      pin(pw[decltype(word)::value]);
    };
    auto step_d = [&](auto word, const uint32_t (&pw)[16]) {
      l = sum2bf(pw[decltype(word)::value], l);
      pin(l);
    };
    auto exp_word = [&](auto word, const f32x16 (&sc)[2], float negm, uint32_t (&pw)[16]) {
      step_f(word, sc, negm);
      step_x();
      step_c(word, pw);
    };
    // slot r of a run of words from w0 on, two slots a word
    auto run_slot = [&](auto r, auto w0, const f32x16 (&sc)[2], float negm, uint32_t (&pw)[16]) {
      constexpr int R = decltype(r)::value, W = decltype(w0)::value + R / 2;
      if constexpr (R % 2 == 0) {
        step_x();
      } else {
        step_c(std::integral_constant<int, W>{}, pw);
        if constexpr (W < 15) step_f(std::integral_constant<int, W + 1>{}, sc, negm);
      }
    };
    auto max_pair = [&](auto pair, const f32x16 (&sc)[2]) {
      constexpr int i = decltype(pair)::value, kt = i >> 3, e = 2 * (i & 7);
      if constexpr (i % 2 == 0) mx = fmaxf(fmaxf(mx, sc[kt][e]), sc[kt][e + 1]);
      else mx1 = fmaxf(fmaxf(mx1, sc[kt][e]), sc[kt][e + 1]);
    };
    // the reference point of the exponentials follows the running maximum only when some row's maximum has grown by more
    // than 2^8: O and lse do not depend on it. O is scaled after the product that is under way.
    float alpha = 1.f;
    auto follow_max = [&]() -> bool {
      mx = max_halves(fmaxf(mx, mx1));
      const bool grow = __builtin_amdgcn_ballot_w64((mx - m) * sl2 > 8.0f) != 0;
      if (grow) {
        alpha = fast_exp2((m - mx) * sl2);
        m = mx;
        l *= alpha;
      }
      return grow;
    };
    auto rescale = [&]() {
#pragma unroll
      for (int i = 0; i < NDT; ++i)
#pragma unroll
        for (int e = 0; e < 16; ++e) oacc[i][e] *= alpha;
    };
    auto mask = [&](int tile, f32x16 (&sc)[2]) {
      const int kbase = opaque(tile * 64 + lh * 4 - (qw0 + lr));  // key - q for element (kt, e) is kbase + kt*32 + (e>>2)*8 + (e&3)
#pragma unroll
      for (int kt = 0; kt < 2; ++kt)
#pragma unroll
        for (int e = 0; e < 16; ++e) sc[kt][e] = (kbase + kt * 32 + (e >> 2) * 8 + (e & 3) > 0) ? -INFINITY : sc[kt][e];
    };
    // Tile t (parity par): its words 4 .. 11 run under the next tile's scores, words 12 .. 15, the next tile's row maximum and its
    // words 0 .. 3 under O += P V. The dot products of the row sum need the matrix pipe and go together where it is free.
    // One barrier per tile: past it tile t + 1's K and tile t's V are in LDS and the buffers of K t and V t - 1 are free.
    constexpr std::integral_constant<int, 0> c0{};
    constexpr std::integral_constant<int, 4> c4{};
    auto full_tile = [&](auto par, int t, f32x16 (&sc)[2], f32x16 (&sn)[2], uint32_t (&pc)[16], uint32_t (&pn)[16]) {
      tile_barrier();
      slots<0, AH>([&](auto i) { request(par, i); });
      const int tk = t + 2 < n ? t + 2 : n - 1;
      const uint8_t* kr = kp + (long)tk * 64 * kst;
      const uint8_t* vr = vp + (long)(t + 1) * 64 * vst;
      uint8_t* kd = lds + decltype(par)::value * TILE;
      uint8_t* vd = lds + (2 + (decltype(par)::value ^ 1)) * TILE;
      float negm = -m * sl2;
      mx = m;
      mx1 = m;
      slots<0, 4>([&](auto i) { step_d(i, pc); });
      slot_end();
      slots<0, NA>([&](auto i) {
        constexpr int x = decltype(i)::value;
        score_slot(i, sn);
        request(par, std::integral_constant<int, x + AH>{});
        if constexpr (x < 4) lk.issue_one(x, kr, kst, kd);
        else if constexpr (x < 8) lv.issue_one(x - 4, vr, vst, vd);
        run_slot(i, c4, sc, negm, pc);
        if constexpr (x >= 9) max_pair(std::integral_constant<int, x - 9>{}, sn);
        slot_end();
      });
      if (t + 1 == last) {
        mask(t + 1, sn);
        mx = m;
        mx1 = m;
        slots<0, 7>([&](auto j) { max_pair(j, sn); });
      }
      slots<0, 8>([&](auto i) {
        constexpr int x = decltype(i)::value;
        out_slot(i, pc);
        request(par, std::integral_constant<int, x + AH + NA>{});
        run_slot(std::integral_constant<int, x + NA>{}, c4, sc, negm, pc);
        if constexpr (x == 0) max_pair(std::integral_constant<int, 7>{}, sn);
        if constexpr (x >= 2 && x < 6) slots<2 * x + 4, 2 * x + 6>([&](auto j) { max_pair(j, sn); });
        slot_end();
      });
      slots<4, 16>([&](auto i) { step_d(i, pc); });
      const bool grow = follow_max();
      negm = -m * sl2;
      step_f(c0, sn, negm);
      slots<8, NB>([&](auto i) {
        constexpr int x = decltype(i)::value;
        out_slot(i, pc);
        request(par, std::integral_constant<int, x + AH + NA>{});
        run_slot(std::integral_constant<int, x - 8>{}, c0, sn, negm, pn);
        slot_end();
      });
      if (grow) rescale();
    };
    // the wavefront's last tile: no scores to make
    auto last_tile = [&](auto par, f32x16 (&sc)[2], uint32_t (&pc)[16]) {
      const float negm = -m * sl2;
      slots<NA, NA + AH>([&](auto i) { request(par, i); });
      slots<4, 8>([&](auto i) { exp_word(i, sc, negm, pc); });
      slot_end();
      slots<0, NB>([&](auto i) {
        constexpr int x = decltype(i)::value;
        out_slot(i, pc);
        request(par, std::integral_constant<int, x + AH + NA>{});
        if constexpr (x < 8) exp_word(std::integral_constant<int, x + 8>{}, sc, negm, pc);
        slot_end();
      });
      slots<0, 16>([&](auto i) { step_d(i, pc); });
    };

    constexpr std::integral_constant<int, 0> even{};
    constexpr std::integral_constant<int, 1> odd{};
    asm volatile("s_waitcnt vmcnt(8)\n\ts_barrier" ::: "memory");  // tile t0's K
    slots<0, AH>([&](auto i) { request(odd, i); });
    slots<0, NA>([&](auto i) {
      constexpr int x = decltype(i)::value;
      if constexpr (x % 2 == 0) landed<(x + AH <= NA ? AH - 2 : NA - 2 - x)>(kf[x], kf[x + 1]);
      const bf16x8 f = kf[x].get();
      if constexpr (x % NKS == 0) scA[x / NKS] = mfma_bf16(f, qf[0], f32x16{});
      else scA[x / NKS] = mfma_bf16(f, qf[x % NKS], scA[x / NKS]);
      if constexpr (x + AH < NA) request(odd, std::integral_constant<int, x + AH>{});
      slot_end();
    });
    if (t0 == last) mask(t0, scA);
    mx = m;
    mx1 = m;
    slots<0, 16>([&](auto i) { max_pair(i, scA); });
    follow_max();  // (O is zero)
    slots<0, 4>([&](auto i) { exp_word(i, scA, -m * sl2, pA); });
    step_f(c4, scA, -m * sl2);
    for (int t = t0; t + 2 < n; t += 2) {
      full_tile(even, t, scA, scB, pA, pB);
      full_tile(odd, t + 1, scB, scA, pB, pA);
    }
    if (wave >= 2) {
      full_tile(even, n - 2, scA, scB, pA, pB);
      tile_barrier();
      last_tile(odd, scB, pB);
    } else {   // (V of the last tile is loaded for the others)
      tile_barrier();
      issue_v(n - 1);
      last_tile(even, scA, pA);
      tile_barrier();
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");  // no load into LDS is on its way when it is given back (both ways have waited)

    const int myq = qw0 + lr;
    const float lt = l + __shfl_xor(l, 32, 64);
    const float inv = 1.0f / lt;
#pragma unroll
    for (int dt = 0; dt < NDT; ++dt)
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int d = dt * 32 + 8 * j + 4 * lh;
        u32x2 w = {pack2bf(oacc[dt][4 * j] * inv, oacc[dt][4 * j + 1] * inv),
                   pack2bf(oacc[dt][4 * j + 2] * inv, oacc[dt][4 * j + 3] * inv)};
        *(u32x2*)(op + (long)myq * o.st + d) = w;
      }
    if (lh == 0) lse[(long)bh * T + myq] = (m * sl2 + log2f(lt)) * LN2;  // m is the raw-score maximum
    if (pass + 1 < npass) __syncthreads();  // the stages are free for the partner block
  }
}

// =========================================================================================== dQ
template <int D>
__global__ __launch_bounds__(256, 2) void attnD_dq_kernel(AttnT q, AttnT k, AttnT v, AttnT go, AttnT dq,
                                                                        float* __restrict__ stats, long rows, int T, int H,
                                                                        float scale, float sl2, int nw, int turn, AttnT o,
                                                                        const float* __restrict__ lse) {
  typedef Geo<D> G;
  constexpr int TILE = G::TILE, NKS = G::NKS, NDT = G::NDT;
  constexpr int AH = 4;  // fragments asked for ahead of their MFMA: from slot 20 on, behind the barrier, the next half's
  static_assert(NKS == 8 && NDT == 4, "three phases of eight slots");
  __shared__ __attribute__((aligned(1024))) uint8_t lds[4 * TILE];  // K even, K odd, V even, V odd tile
  const int tid = threadIdx.x, lane = tid & 63, lr = lane & 31, lh = lane >> 5;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  int bx, bh;
  xcd_block(T / 128, gridDim.y, bx, bh, turn);
  const int b = bh / H, h = bh % H;
  const bf16_t* qp = q.p + b * q.sb + h * q.sh;
  const bf16_t* gp = go.p + b * go.sb + h * go.sh;
  const uint8_t* kp = (const uint8_t*)(k.p + b * k.sb + h * k.sh);
  const uint8_t* vp = (const uint8_t*)(v.p + b * v.sb + h * v.sh);
  const int nx = T / 128, npass = paired_passes(nx);
  const long kst = k.st * 2, vst = v.st * 2;
  TileLoad<D, 16 / G::TPI> lk, lv;
  lk.init(kst, wave, lane);
  lv.init(vst, wave, lane);
  auto issue_k = [&](int tile) { lk.issue(kp + (long)tile * 64 * kst, kst, lds + (tile & 1) * TILE); };
  auto issue_v = [&](int tile) { lv.issue(vp + (long)tile * 64 * vst, vst, lds + (2 + (tile & 1)) * TILE); };
  FragAddr<D> fa;
  fa.init((uint32_t)(uintptr_t)(lds_void_t*)lds, lane);
  for (int pass = 0; pass < npass; ++pass) {
    const int qb = paired_block(nx, bx, pass, true);
    const int q0 = qb * 128, qw0 = q0 + wave * 32, myq = qw0 + lr;
    const int n = (q0 + 128) / 64;           // even; tiles n - 2 and n - 1 cover the workgroup's own 128 tokens
    const int t0 = band_first_tile(qb, nw);  // even
    issue_k(t0);
    issue_v(t0);
    issue_k(t0 + 1);
    issue_v(t0 + 1);
    bf16x8 qf[NKS], gf[NKS];
#pragma unroll
    for (int s = 0; s < NKS; ++s) {
      qf[s] = *(const bf16x8*)(qp + (long)myq * q.st + 16 * s + 8 * lh);
      gf[s] = *(const bf16x8*)(gp + (long)myq * go.st + 16 * s + 8 * lh);
    }
    // the row statistics of this wavefront's queries, made here (this kernel runs first) and left for dK/dV:
    // -sum_d dO O and -lse / scale
    float myD, myL;
    {
      const bf16_t* orow = o.p + b * o.sb + h * o.sh + (long)myq * o.st;
      float dot = 0.f;
#pragma unroll
      for (int s = 0; s < NKS; ++s) {
        const u32x4 ov = *(const u32x4*)(orow + 16 * s + 8 * lh);
        const u32x4 gv = __builtin_bit_cast(u32x4, gf[s]);
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          dot += bflo(ov[w]) * bflo(gv[w]);
          dot += bfhi(ov[w]) * bfhi(gv[w]);
        }
      }
      dot += __shfl_xor(dot, 32, 64);
      myD = -dot;
      myL = -lse[(long)bh * T + myq] * (1.0f / scale);
    }
    f32x16 dqa[NDT];
#pragma unroll
    for (int i = 0; i < NDT; ++i)
#pragma unroll
      for (int e = 0; e < 16; ++e) dqa[i][e] = 0.f;

    // Half tiles of 32 keys, h = 2 tile + half, at LDS offset (h & 3) TILE / 2. While half h's dS and dQ += dS K are made, half
    // h + 1's S and dP are: 24 slots of one MFMA, S (0 .. 7), dP (8 .. 15), dQ (16 .. 23). The wavefront's last half is the one on
    // its diagonal. One barrier per half, before slot 20: this half's columns have been read and what the half before asked for has
    // landed, so that V t + 2 (K t + 2) may replace V t (K t) behind an even (odd) half's barrier and the next half's rows be read.
    f32x16 Sn, dP;
    uint32_t pw[8], dsw[8];
    float f0, f1;
    RowFrag rf[16];
    ColFrag cf[8];
    constexpr int HALF = 32 * G::ROWB;
    auto request_row = [&](auto slot, uint32_t off) {
      constexpr int i = decltype(slot)::value;
      rf[i].template request<i < 8 ? 0 : 2 * TILE>(fa.rows[i % 8] + off);
    };
    auto request_col = [&](auto slot, uint32_t off) {
      constexpr int i = decltype(slot)::value - 16;
      cf[i].template request<(i / NDT) * 16 * G::ROWB>(fa.lo[i % NDT] + off, fa.hi[i % NDT] + off);
    };
    // LDS instructions issued after fragment i + 1's when slot i waits for the two (0 behind the barrier, which waits for all but those after it)
    auto after = [](int i) constexpr {
      int c = 0;
      for (int x = i + 2; x < i + AH; ++x) c += (x % 24) < 16 ? 1 : 2;
      return c;
    };
    auto row_slot = [&](auto slot, auto aft) {
      constexpr int i = decltype(slot)::value, s = i % 8;
      if constexpr (i % 2 == 0) landed<decltype(aft)::value>(rf[i], rf[i + 1]);
      const bf16x8 f = rf[i].get();
      if constexpr (s == 0) {
        float c = i < 8 ? myL : myD;
        pin(c);  // (spread by moves each time: kept as constant operands the two would take 32 registers)
        f32x16& x = i < 8 ? Sn : dP;
#pragma unroll
        for (int e = 0; e < 16; ++e) x[e] = c;
      }
      if constexpr (i < 8) Sn = mfma_bf16(f, qf[s], Sn);
      else dP = mfma_bf16(f, gf[s], dP);
    };
    auto col_slot = [&](auto slot, auto aft) {
      constexpr int i = decltype(slot)::value - 16, ks = i / NDT, dt = i % NDT;
      if constexpr (i % 2 == 0) landed<decltype(aft)::value>(cf[i], cf[i + 1]);
      const bf16x8 f = cf[i].get();
      dqa[dt] = mfma_bf16(f, frag_from(dsw[4 * ks], dsw[4 * ks + 1], dsw[4 * ks + 2], dsw[4 * ks + 3]), dqa[dt]);
    };
    auto ds_word = [&](auto word) {  // the reference multiplies dP - delta by the rounded P
      constexpr int w = decltype(word)::value;
      dsw[w] = pack2bf(bflo(pw[w]) * dP[2 * w], bfhi(pw[w]) * dP[2 * w + 1]);
      pin(dsw[w]);
    };
    auto step_f = [&](auto word) {
      constexpr int w = decltype(word)::value;
      f0 = Sn[2 * w] * sl2;
      f1 = Sn[2 * w + 1] * sl2;
      pin(f0, f1);
    };
    auto step_x = [&]() {
      f0 = fast_exp2(f0);
      f1 = fast_exp2(f1);
      pin(f0, f1);
    };
    auto step_c = [&](auto word) {
      pw[decltype(word)::value] = pack2bf(f0, f1);
      pin(pw[decltype(word)::value]);
    };
    auto mask = [&]() {  // Sn is the wavefront's diagonal
      const int kbase = opaque(lh * 4 - lr);
#pragma unroll
      for (int e = 0; e < 16; ++e) Sn[e] = (kbase + (e >> 2) * 8 + (e & 3) > 0) ? -INFINITY : Sn[e];
    };

    const int h0 = 2 * t0, hl = 2 * (n - 2) + wave;
    tile_barrier();
    // half h0's S, dP and P
    slots<0, AH>([&](auto i) { request_row(i, 0u); });
    slots<0, 16>([&](auto i) {
      constexpr int x = decltype(i)::value;
      row_slot(i, std::integral_constant<int, (x + AH <= 16 ? AH - 2 : 14 - x) < 0 ? 0 : (x + AH <= 16 ? AH - 2 : 14 - x)>{});
      if constexpr (x + AH < 16) request_row(std::integral_constant<int, x + AH>{}, 0u);
      slot_end();
    });
    if (h0 == hl) mask();
    slots<0, 8>([&](auto i) {
      step_f(i);
      step_x();
      step_c(i);
    });
    slots<0, AH>([&](auto i) { request_row(i, (uint32_t)HALF); });
    for (int hh = h0; hh < hl; ++hh) {
      const uint32_t roff = ((hh + 1) & 3) * HALF, coff = (hh & 3) * HALF, noff = ((hh + 2) & 3) * HALF;
      slot_end();
      slots<0, 8>([&](auto i) {
        constexpr int x = decltype(i)::value;
        row_slot(i, std::integral_constant<int, after(x)>{});
        request_row(std::integral_constant<int, x + AH>{}, roff);
        ds_word(i);
        slot_end();
      });
      row_slot(std::integral_constant<int, 8>{}, std::integral_constant<int, after(8)>{});
      request_row(std::integral_constant<int, 8 + AH>{}, roff);
      if (hh + 1 == hl) mask();
      step_f(std::integral_constant<int, 0>{});
      slot_end();
      const int lt = (hh >> 1) + 2 < n ? (hh >> 1) + 2 : n - 1;
      const bool odd = hh & 1;
      const uint8_t* lp = odd ? kp + (long)lt * 64 * kst : vp + (long)lt * 64 * vst;
      const long lst = odd ? kst : vst;
      uint8_t* ld = lds + (odd ? 0 : 2 * TILE) + ((hh >> 1) & 1) * TILE;
      slots<9, 24>([&](auto i) {
        constexpr int x = decltype(i)::value;
        if constexpr (x == 20) {
          asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");
          slot_end();
        }
        constexpr int aft = x < 20 ? after(x) : AH;  // (already there)
        if constexpr (x < 16) row_slot(i, std::integral_constant<int, after(x)>{});
        else col_slot(i, std::integral_constant<int, aft>{});
        if constexpr (x + AH < 16) request_row(std::integral_constant<int, x + AH>{}, roff);
        else if constexpr (x + AH < 24) request_col(std::integral_constant<int, x + AH>{}, coff);
        else request_row(std::integral_constant<int, x + AH - 24>{}, noff);
        if constexpr (x >= 20) (odd ? lk : lv).issue_one(x - 20, lp, lst, ld);
        if constexpr (x % 2 == 1) {
          step_x();
        } else {
          step_c(std::integral_constant<int, (x - 10) / 2>{});
          step_f(std::integral_constant<int, (x - 8) / 2>{});
        }
        slot_end();
      });
      step_c(std::integral_constant<int, 7>{});
    }
    // the wavefront's last half
    {
      const uint32_t coff = (hl & 3) * HALF;
      asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // (the rows asked for are not used)
      slots<0, AH>([&](auto i) { if constexpr (decltype(i)::value % 2 == 0) landed<0>(rf[decltype(i)::value], rf[decltype(i)::value + 1]); });
      slots<16, 16 + AH>([&](auto i) { request_col(i, coff); });
      slots<0, 8>([&](auto i) { ds_word(i); });
      slot_end();
      slots<16, 24>([&](auto i) {
        constexpr int x = decltype(i)::value;
        col_slot(i, std::integral_constant<int, x % 2 ? 0 : 2 * (x + AH <= 24 ? AH - 2 : 22 - x)>{});
        if constexpr (x + AH < 24) request_col(std::integral_constant<int, x + AH>{}, coff);
        slot_end();
      });
    }
    // The other wavefronts' halves. They read what this one's last loads bring (the first wavefront's share of the last K tile): those have
    // to have landed before its next barrier. (Without the wait rare launches had 45 of a block's rows of dQ wrong.)
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    for (int x = wave; x < 3; ++x) asm volatile("s_barrier" ::: "memory");
    bf16_t* dqp = dq.p + b * dq.sb + h * dq.sh + (long)myq * dq.st;
    store_grad_row<D>(dqa, scale, dqp, lh);
    if (lh == 0) {
      stats[(long)bh * T + myq] = myD;
      stats[rows + (long)bh * T + myq] = myL;
    }
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
    if (pass + 1 < npass) __syncthreads();  // the stages are free for the partner block
  }
}

template <int D>
int fwd_launch(const void* q, const long* qs, const void* k, const long* ks, const void* v, const long* vs, void* o,
               const long* os, float* lse, int B, int H, int T, float scale, int nw, hipStream_t s) {
  if (tfb_attn_fwd_pair_applies(D, T, (long)B * H, nw, ks, vs)) return tfb_attn_fwd_pair_impl(q, qs, k, ks, v, vs, o, os, lse, B, H, T, D, scale, nw, s);
  hipLaunchKernelGGL(attnD_fwd_kernel<D>, dim3(paired_grid(T / 128, B * H, 2), B * H), dim3(256), 0, s, mk(q, qs), mk(k, ks), mk(v, vs),
                     mk(o, os), lse, T, H, scale * LOG2E, nw, first_round(T / 128, B * H, true));
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}
template <int D>
int bwd_launch(const void* q, const long* qs, const void* k, const long* ks, const void* v, const long* vs, const void* o,
               const long* os, const void* go, const long* gos, void* dq, const long* dqs, void* dk, const long* dks, void* dv,
               const long* dvs, const float* lse, float* stats, int B, int H, int T, float scale, int nw, hipStream_t s) {
  const long rows = (long)B * H * T;
  if (tfb_attn_dq_pair_applies(D, T, (long)B * H, nw, ks, vs)) {
    const int st = tfb_attn_dq_pair_impl(q, qs, k, ks, v, vs, o, os, go, gos, dq, dqs, lse, stats, B, H, T, D, scale, nullptr, nullptr, nw, s);
    if (st != TFB_OK) return st;
  } else {
    hipLaunchKernelGGL(attnD_dq_kernel<D>, dim3(paired_grid(T / 128, B * H, 2), B * H), dim3(256), 0, s, mk(q, qs), mk(k, ks), mk(v, vs),
                       mk(go, gos), mk(dq, dqs), stats, rows, T, H, scale, scale * LOG2E, nw, first_round(T / 128, B * H, true), mk(o, os), lse);
    TFB_LAUNCH_CHECK();
  }
  return tfb_attn_dkdv_impl(q, qs, k, ks, v, vs, go, gos, dk, dks, dv, dvs, stats, B, H, T, D, scale, nullptr, nullptr, nw, s);
}

}  // namespace

// Called by tfb_attn_fwd / tfb_attn_bwd for D = 128 (arguments validated there: T % 128 == 0, strides % 8 == 0).
int tfb_attn128_fwd_impl(const void* q, const long* qs, const void* k, const long* ks, const void* v, const long* vs,
                       void* o, const long* os, float* lse, int B, int H, int T, float scale, int nw, hipStream_t s) {
  return fwd_launch<128>(q, qs, k, ks, v, vs, o, os, lse, B, H, T, scale, nw, s);
}
// stats: fp32 [2][B*H][T] scratch (-delta, then -lse / scale), written by the dQ kernel and read by dK/dV.
int tfb_attn128_bwd_impl(const void* q, const long* qs, const void* k, const long* ks, const void* v, const long* vs,
                       const void* o, const long* os, const void* go, const long* gos, void* dq, const long* dqs, void* dk,
                       const long* dks, void* dv, const long* dvs, const float* lse, float* stats, int B, int H, int T,
                       float scale, int nw, hipStream_t s) {
  return bwd_launch<128>(q, qs, k, ks, v, vs, o, os, go, gos, dq, dqs, dk, dks, dv, dvs, lse, stats, B, H, T, scale, nw, s);
}
