// Loss head: softcap + log-softmax + cross-entropy on bf16 logits, and the LM-head GEMM with the
// log-sum-exp fused into its epilogue.
//
// Replaces _loss_fwd_kernel / _loss_bwd_kernel behind fused_loss(logits, targets, reduction, softcap)
// (round1/source/train.py:4543, 4584, 4691; eager form 4481-4495), the row-weighted form of
// round2/source/train.py:6364-6391 (ignore_index -1 = weight 0), and the lm_head matmul in front of
// them (round1/source/train.py:8668, 9191-9212).
//
// Math per row, fp32 from the bf16-rounded logits x: s_v = c tanh(x_v / c) (or s_v = x_v without a
// softcap), lse = log sum_v exp(s_v), loss = lse - s_target; d x_v = g (softmax_v - [v = target])
// (1 - tanh^2). Only lse is saved; the backward recomputes tanh / exp.
//
// lmhead_fwd is the GEMM logits = x @ W^T (W [V, d]) whose epilogue rounds each accumulator to bf16,
// stores it, and reduces exp(s - shift) over the 64 vocabulary columns a wavefront holds for each row
// (in registers: a lane owns 32 of them, its partner lane the rest) into a [rows][V/64] table of
// (max, sum) pairs; a finishing kernel merges a row's pairs, reads the target logit and writes lse and
// the row loss. Launches large enough for the persistent 256 x 256 kernel take that instead, and a pass over the logits it wrote.
#include "gemm_ring.hpp"

namespace {

__device__ __forceinline__ float fexp(float x) { return __builtin_amdgcn_exp2f(x * 1.4426950408889634f); }

// 1 / (exp(2 y) + 1), correctly rounded: a Newton step on the hardware's reciprocal, which is off by one ulp at most, gives the
// bits of an IEEE division at a third of its instructions, for each of the 201,326,592 floats from 1 to 2^24 (compared one by one on
// gfx950; the tests compare the gradient of every bf16 logit); beyond, tanh is 1 either way. The clamp keeps the Newton step from
// inf * 0; it is the minimum that hands a NaN on (one instruction, as fminf, which would make a NaN logit's tanh 1).
__device__ __forceinline__ float tanh_rcp(float y) {
  const float d = __builtin_elementwise_minimum(__builtin_amdgcn_exp2f(y * 2.8853900817779268f), 0x1p100f) + 1.0f;
  const float r = __builtin_amdgcn_rcpf(d);
  return __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
}
// tanh(y) = 1 - 2 / (exp(2 y) + 1) (doubling is exact: the fma has the bits of the product and the difference)
__device__ __forceinline__ float tanh_fast(float y) { return __builtin_fmaf(-2.0f, tanh_rcp(y), 1.0f); }

struct MS {
  float m, s;
};
__device__ __forceinline__ MS ms_merge(MS a, MS b) {
  float m = fmaxf(a.m, b.m);
  MS r;
  r.m = m;
  r.s = a.s * fexp(a.m - m) + b.s * fexp(b.m - m);
  return r;
}

// ------------------------------------------------------------------------------------ row weights
// One workgroup: w[i] = valid_i / max(1, #valid) for the mean over the rows that count (mean != 0), else valid_i; a row
// counts when 0 <= t_i < V (V <= 0: when 0 <= t_i): the rows the loss kernels give a loss to.
template <typename IDX>
__global__ __launch_bounds__(1024) void loss_row_weights_kernel(const IDX* __restrict__ tg, float* __restrict__ w, long rows,
                                                               int mean, long V) {
  auto valid = [&](IDX t) { return t >= 0 && (long)t < V; };
  __shared__ int cnt[16];
  float each = 1.0f;
  if (mean) {
    int c = 0;
    for (long i = threadIdx.x; i < rows; i += 4096) {
      IDX t[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) t[k] = i + 1024 * k < rows ? tg[i + 1024 * k] : (IDX)-1;
#pragma unroll
      for (int k = 0; k < 4; ++k) c += valid(t[k]);
    }
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) c += __shfl_xor(c, o);
    if ((threadIdx.x & 63) == 0) cnt[threadIdx.x >> 6] = c;
    __syncthreads();
    int n = 0;
#pragma unroll
    for (int k = 0; k < 16; ++k) n += cnt[k];
    each = 1.0f / (float)(n > 1 ? n : 1);
  }
  for (long i = threadIdx.x; i < rows; i += 1024) w[i] = valid(tg[i]) ? each : 0.f;
}

// ------------------------------------------------------------------------------------ loss on logits
// A row belongs to TPR threads: a workgroup of 256, or a wavefront (four rows a workgroup) where V <= 2048, whose rows would
// leave half of a workgroup or more without a value (16384 x 1024, in place: 39 us with a workgroup a row, 20 with a wavefront).
constexpr int WAVE_ROW_V = 2048;

// exp(cap tanh(x / cap) - cap). (exp2(-2 cap log2(e) / (exp(2 x / cap) + 1)) needs two instructions less; but the error of its
// reciprocal and of the inner exponential counts 2 cap times over: the mean error of lse over 9600 rows x 8192 of deviation
// 0.5, cap = 30, is then 0.42e-6 with the hardware's reciprocal and 0.61e-6 with an exact one, 0.16e-6 this way. exp2(fma(t, k, -k)) with
// k = cap log2(e) needs two less as well, and takes 2 % off the pass; but the rounding of k has one sign for all terms of a row: 9600 x 8192 of
// deviation 2, cap = 15, 0.32e-6 this way and 0.46e-6 so.)
__device__ __forceinline__ float capped_exp(float x, float icap, float cap) { return fexp(cap * tanh_fast(x * icap) - cap); }

// The pair (max, sum exp) of eight logits joined to a (with a softcap cap is the maximum: it bounds every value).
__device__ __forceinline__ void ms_add8(MS& a, const u32x4& u, float icap, float cap) {
  float v[8];
  unpack8bf(u, v);
  if (cap > 0.f) {
#pragma unroll
    for (int k = 0; k < 8; ++k) a.s += capped_exp(v[k], icap, cap);
  } else {
    float mx = a.m, t = 0.f;
#pragma unroll
    for (int k = 0; k < 8; ++k) mx = fmaxf(mx, v[k]);
    const float sc = fexp(a.m - mx);
#pragma unroll
    for (int k = 0; k < 8; ++k) t += fexp(v[k] - mx);
    a.s = a.s * sc + t;
    a.m = mx;
  }
}

// Evaluation: four chunks with one running maximum for their 32 values. Chunks beyond V hold -inf; i, step: the first chunk's
// place in the row and the distance of two.
__device__ __forceinline__ void ms_add32(MS& a, const u32x4* u, int i, int step, int V, float icap, float cap) {
  if (cap > 0.f) {
#pragma unroll
    for (int c = 0; c < 4; ++c)
      if (i + step * c < V) {
#pragma unroll
        for (int k = 0; k < 4; ++k) a.s += capped_exp(bflo(u[c][k]), icap, cap) + capped_exp(bfhi(u[c][k]), icap, cap);
      }
  } else {
    float mx = a.m, t = 0.f;
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) mx = fmaxf(fmaxf(mx, bflo(u[c][k])), bfhi(u[c][k]));
#pragma unroll
    for (int c = 0; c < 4; ++c)
#pragma unroll
      for (int k = 0; k < 4; ++k) t += fexp(bflo(u[c][k]) - mx) + fexp(bfhi(u[c][k]) - mx);
    a.s = a.s * fexp(a.m - mx) + t;
    a.m = mx;
  }
}
__device__ __forceinline__ u32x4 logits8(const bf16_t* x, int i, int V) {
  return i < V ? *(const u32x4*)(x + i) : u32x4{0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u};
}
__device__ __forceinline__ MS ms_wave(MS a) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) a = ms_merge(a, MS{__shfl_xor(a.m, o, 64), __shfl_xor(a.s, o, 64)});
  return a;
}
// A workgroup's row: the pair of all, in its first thread.
__device__ __forceinline__ MS ms_group(MS a, float (&rm)[4], float (&rs)[4]) {
  a = ms_wave(a);
  if ((threadIdx.x & 63) == 0) {
    rm[threadIdx.x >> 6] = a.m;
    rs[threadIdx.x >> 6] = a.s;
  }
  __syncthreads();
  if (threadIdx.x == 0)
    for (int i = 1; i < 4; ++i) a = ms_merge(a, MS{rm[i], rs[i]});
  return a;
}
// A wavefront's row of at most four chunks a lane, in all lanes: every chunk is what one wavefront of a workgroup would hold, and
// they are joined in that order, so the row's lse has the same bits whichever way it is taken.
__device__ __forceinline__ MS ms_wave_row(const u32x4 (&u)[4], int t0, int V, float icap, float cap) {
  const MS none{cap > 0.f ? cap : -1e30f, 0.f};
  MS a = none;
#pragma unroll
  for (int c = 0; c < 4; ++c) {
    if (c && 512 * c >= V) break;   // (a chunk that no lane has would change nothing)
    MS b = none;
    if ((t0 + 64 * c) * 8 < V) ms_add8(b, u[c], icap, cap);
    b = ms_wave(b);
    a = c ? ms_merge(a, b) : b;
  }
  return a;
}
// d x_v = g (softmax_v - [v == t]) (1 - tanh^2) of eight values from v = i on; t: the row's target, -1 where it has none.
// The target's one is taken off behind a branch that a wavefront takes for one of its chunks at most: a comparison, a select and a
// subtraction for each value were a quarter of the vector instructions that these passes spend their time on beside memory.
__device__ __forceinline__ u32x4 loss_grad8(const u32x4& u, int i, int t, float g, float l, float icap, float cap) {
  float v[8], d[8];
  unpack8bf(u, v);
  if (cap > 0.f) {
#pragma unroll
    for (int k = 0; k < 8; ++k) {
      v[k] = tanh_fast(v[k] * icap);
      d[k] = fexp(cap * v[k] - l);
    }
  } else {
#pragma unroll
    for (int k = 0; k < 8; ++k) d[k] = fexp(v[k] - l);
  }
  if ((unsigned)(t - i) < 8u) {
#pragma unroll
    for (int k = 0; k < 8; ++k) d[k] = t - i == k ? d[k] - 1.0f : d[k];
  }
#pragma unroll
  for (int k = 0; k < 8; ++k) d[k] *= g;
  if (cap > 0.f) {
#pragma unroll
    for (int k = 0; k < 8; ++k) d[k] *= 1.0f - v[k] * v[k];
  }
  return u32x4{pack2bf(d[0], d[1]), pack2bf(d[2], d[3]), pack2bf(d[4], d[5]), pack2bf(d[6], d[7])};
}

// The same bits with a softcap, one value after the other. Where a launch keeps the SIMDs full, eight values' exponentials and reciprocals side by
// side only wait for one another, and the target's one is then a twelfth of the instructions; a short launch has the row's end to wait for. us,
// cap = 15, side by side -> each (from 2048 blocks on, eight for each CU): rows of 8192, 128 of them 5.8 -> 6.8, 1024 14.5 -> 15.1, 2048 24.3 -> 24.1, 8192 77.7 -> 74.8, 16384 146 -> 139; of 1024, 2048
// of them 6.4 -> 6.5, 16384 28.4 -> 27.5; the backward alone, of 8192, 128 of them 4.5 -> 5.5, 1024 9.6 -> 9.9, 8192 46.0 -> 44.5.
__device__ __forceinline__ u32x4 loss_grad8_each(const u32x4& u, int i, int t, float g, float l, float icap, float cap) {
  float d[8];
#pragma unroll
  for (int k = 0; k < 8; ++k) {
    const float x = k & 1 ? bfhi(u[k >> 1]) : bflo(u[k >> 1]), hot = i + k == t ? 1.0f : 0.0f;
    if (cap > 0.f) {  // (always; the branch is what keeps the values apart)
      const float th = tanh_fast(x * icap);
      d[k] = g * (fexp(cap * th - l) - hot) * (1.0f - th * th);
    } else {
      d[k] = g * (fexp(x - l) - hot);
    }
  }
  return u32x4{pack2bf(d[0], d[1]), pack2bf(d[2], d[3]), pack2bf(d[4], d[5]), pack2bf(d[6], d[7])};
}
static inline bool loss_each(long blocks, float softcap) { return softcap > 0.f && blocks >= 2048; }

// loss_row = w * (lse - s_t) with w = row_w[row] (or 1), 0 for a target outside [0, V). Bound by memory: four 16-byte loads a
// lane in flight. EVAL: the pass over the LM head's logits where the GEMM leaves it to one.
template <typename IDX, int TPR, bool EVAL>
__global__ __launch_bounds__(256) void loss_fwd_kernel(const bf16_t* __restrict__ x, const IDX* __restrict__ tg,
                                                      const float* __restrict__ row_w, float* __restrict__ loss,
                                                      float* __restrict__ lse, long rows, int V, float cap) {
  __shared__ float rm[4], rs[4];
  const long row = (long)blockIdx.x * (256 / TPR) + threadIdx.x / TPR;
  if (TPR < 256 && row >= rows) return;
  const bf16_t* xr = x + row * V;
  const int t0 = threadIdx.x % TPR;
  const float icap = cap > 0.f ? 1.0f / cap : 0.f;
  MS a{cap > 0.f ? cap : -1e30f, 0.f};
  for (int i0 = t0 * 8; i0 < V || (TPR == 64 && i0 == t0 * 8); i0 += 4 * TPR * 8) {   // (a wavefront's row is one turn of all its lanes)
    u32x4 u[4];
#pragma unroll
    for (int c = 0; c < 4; ++c) u[c] = logits8(xr, i0 + TPR * 8 * c, V);
    if constexpr (EVAL) {
      ms_add32(a, u, i0, TPR * 8, V, icap, cap);
    } else if constexpr (TPR == 64) {
      a = ms_wave_row(u, t0, V, icap, cap);
    } else {
#pragma unroll
      for (int c = 0; c < 4; ++c)
        if (i0 + TPR * 8 * c < V) ms_add8(a, u[c], icap, cap);
    }
  }
  if constexpr (TPR == 256) a = ms_group(a, rm, rs);
  else if constexpr (EVAL) a = ms_wave(a);
  if (t0 == 0) {
    const float l = a.m + logf(a.s);
    lse[row] = l;
    const long tt = (long)tg[row];
    float out = 0.f;
    if ((unsigned long)tt < (unsigned long)V) {  // a target outside [0, V) is an ignored row, never an address
      const float xt = bf2f(xr[tt]);
      out = (l - (cap > 0.f ? cap * tanh_fast(xt * icap) : xt)) * (row_w ? row_w[row] : 1.0f);
    }
    loss[row] = out;
  }
}

// g_row = grow[row] (upstream grad x row weight); a target outside [0, V) -> 0.
template <typename IDX, int TPR, bool EACH>
__global__ __launch_bounds__(256) void loss_bwd_kernel(const bf16_t* __restrict__ x, const IDX* __restrict__ tg,
                                                      const float* __restrict__ lse, const float* __restrict__ grow,
                                                      bf16_t* __restrict__ dx, long rows, int V, float cap) {
  const long row = (long)blockIdx.x * (256 / TPR) + threadIdx.x / TPR;
  if (TPR < 256 && row >= rows) return;
  const bf16_t* xr = x + row * V;
  bf16_t* dr = dx + row * V;
  const int t0 = threadIdx.x % TPR;
  const long tt = (long)tg[row];
  const bool valid = (unsigned long)tt < (unsigned long)V;  // out of range = ignored
  const float g = valid ? grow[row] : 0.f;
  const int t = valid ? (int)tt : -1;   // (t - i of a chunk at i >= 0 is then no column of it)
  const float l = lse[row];
  const float icap = cap > 0.f ? 1.0f / cap : 0.f;
  // (the next chunk is requested before this chunk's store: a wait for loaded data also waits for every older store)
  u32x4 unext = logits8(xr, t0 * 8, V);
  for (int i = t0 * 8; i < V; i += TPR * 8) {
    const u32x4 u = unext;
    unext = logits8(xr, i + TPR * 8, V);
    *(u32x4*)(dr + i) = EACH ? loss_grad8_each(u, i, t, g, l, icap, cap) : loss_grad8(u, i, t, g, l, icap, cap);
  }
}

// loss_fwd_kernel and loss_bwd_kernel for grow = row_w in ONE pass over the logits: the threads of a row keep it in registers
// (NCH chunks of eight values per thread, V <= 8 TPR NCH), reduce it to lse in the order of loss_fwd_kernel, write lse and
// the weighted row loss, and overwrite the row with d x_v = w (softmax_v - [v = t]) (1 - tanh^2): the gradient for an
// upstream gradient of one, which the caller's two gradient GEMMs scale by the real one. The logits are read once and
// written once where the two kernels read them twice; values equal theirs bit for bit.
// Bound by memory and by the vector instructions beside it. The target's one behind a branch (loss_grad8) and a store that does not pass
// through the caches: rows of 32768, 32768 of them 935 -> 790 us, 8192 249 -> 211, 2048 76 -> 66. A row of 32 chunks is unpacked twice, behind an
// empty asm statement: kept unpacked, its 256 values spilled (4096 rows of 50304 431 us; with the branch alone 257, so 183). With 16 chunks the
// registers suffice: without a softcap two wavefronts a SIMD that unpack once stream better than four that unpack twice (32768 rows 790 us to 860,
// 2048 66 to 64); with one, the four hide more of the exponentials (rows of 32768, cap = 15: 2048 84.0 -> 78.8, 16384 588 -> 532; up to 1024 alike).
// The kernel of 32 chunks is 70 KB of code, more than the instruction cache holds, and moves by up to 8 % with its place in the library.
// EACH: loss_grad8_each. TWICE: unpacked twice.
template <typename IDX, int NCH, int TPR, bool EACH, bool TWICE>
__global__ __launch_bounds__(256) void loss_fwd_bwd_kernel(bf16_t* x, const IDX* __restrict__ tg, const float* __restrict__ row_w,
                                                          float* __restrict__ loss, float* __restrict__ lse, long rows, int V, float cap) {
  __shared__ float rm[4], rs[4], lsh;
  const long row = (long)blockIdx.x * (256 / TPR) + threadIdx.x / TPR;
  if (TPR < 256 && row >= rows) return;
  bf16_t* xr = x + row * V;
  const int t0 = threadIdx.x % TPR;
  const float icap = cap > 0.f ? 1.0f / cap : 0.f;
  u32x4 u[NCH];
#pragma unroll
  for (int j = 0; j < NCH; ++j) u[j] = logits8(xr, (t0 + j * TPR) * 8, V);
  const long tt = (long)tg[row];
  const bool valid = (unsigned long)tt < (unsigned long)V;  // a target outside [0, V) is an ignored row, never an address
  const int t = valid ? (int)tt : -1;
  const float w = valid ? (row_w ? row_w[row] : 1.0f) : 0.f;
  const float xt = valid ? bf2f(xr[tt]) : 0.f;              // (read before any thread overwrites the row)
  MS a{cap > 0.f ? cap : -1e30f, 0.f};
  if constexpr (TPR == 64) {
    a = ms_wave_row(u, t0, V, icap, cap);
  } else {
#pragma unroll
    for (int j = 0; j < NCH; ++j)
      if ((t0 + j * TPR) * 8 < V) ms_add8(a, u[j], icap, cap);
    a = ms_group(a, rm, rs);
  }
  float l = a.m + logf(a.s);
  if (t0 == 0) {
    lse[row] = l;
    loss[row] = valid ? (l - (cap > 0.f ? cap * tanh_fast(xt * icap) : xt)) * w : 0.f;
  }
  if constexpr (TPR == 256) {
    if (t0 == 0) lsh = l;
    __syncthreads();
    l = lsh;
  }
#pragma unroll
  for (int j = 0; j < NCH; ++j) {
    const int i = (t0 + j * TPR) * 8;
    if (TWICE) asm("" : "+v"(u[j]));
    if (i < V) tfb_store_nt((u32x4*)(xr + i), EACH ? loss_grad8_each(u[j], i, t, w, l, icap, cap) : loss_grad8(u[j], i, t, w, l, icap, cap));
  }
}

// ------------------------------------------------------------------------------------ several targets / label smoothing
// loss_row = sum_k rw_k (lse - (1 - eps) s_{t_k} - (eps / V) sum_v s_v), targets tg [K][rows] and weights rw [K][rows]
// (a target < 0 counts with weight 0). K > 1 is the multi-token-prediction loss (round1/source/train.py:4725), eps > 0
// the label-smoothed loss (round2/source/train.py:5697); K = 1, eps = 0 is loss_fwd_kernel with row weights.
// d x_v = g (1 - tanh^2) (W softmax_v - (1 - eps) sum_k rw_k [v = t_k] - W eps / V), W = sum_k rw_k.
constexpr int LOSS_KMAX = 8;

template <typename IDX>
__global__ __launch_bounds__(256) void loss_multi_fwd_kernel(const bf16_t* __restrict__ x, const IDX* __restrict__ tg,
                                                            const float* __restrict__ rw, int K, long rows,
                                                            float* __restrict__ loss, float* __restrict__ lse, int V, float cap,
                                                            float eps) {
  __shared__ float rm[4], rs[4], rt[4];
  const long row = blockIdx.x;
  const bf16_t* xr = x + row * V;
  const float icap = cap > 0.f ? 1.0f / cap : 0.f;
  MS a{-1e30f, 0.f};
  float ssum = 0.f;  // sum_v s_v (label smoothing)
  for (int i = threadIdx.x * 8; i < V; i += 256 * 8) {
    u32x4 u = *(const u32x4*)(xr + i);
    float v[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[2 * k] = bflo(u[k]);
      v[2 * k + 1] = bfhi(u[k]);
    }
    if (cap > 0.f) {
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        const float sv = cap * tanh_fast(v[k] * icap);
        ssum += sv;
        a.s += fexp(sv - cap);
      }
      a.m = cap;
    } else {
      float mx = a.m;
#pragma unroll
      for (int k = 0; k < 8; ++k) mx = fmaxf(mx, v[k]);
      float sc = fexp(a.m - mx), t = 0.f;
#pragma unroll
      for (int k = 0; k < 8; ++k) {
        t += fexp(v[k] - mx);
        ssum += v[k];
      }
      a.s = a.s * sc + t;
      a.m = mx;
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    MS b{__shfl_xor(a.m, o, 64), __shfl_xor(a.s, o, 64)};
    a = ms_merge(a, b);
    ssum += __shfl_xor(ssum, o, 64);
  }
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (lane == 0) {
    rm[wave] = a.m;
    rs[wave] = a.s;
    rt[wave] = ssum;
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    MS t{rm[0], rs[0]};
    for (int i = 1; i < 4; ++i) t = ms_merge(t, MS{rm[i], rs[i]});
    const float l = t.m + logf(t.s);
    const float mean_s = (rt[0] + rt[1] + rt[2] + rt[3]) / (float)V;
    lse[row] = l;
    float out = 0.f;
    for (int k = 0; k < K; ++k) {
      const long tt = (long)tg[(long)k * rows + row];
      if ((unsigned long)tt >= (unsigned long)V) continue;  // negative or beyond the vocabulary: weight 0
      const float xt = bf2f(xr[tt]);
      const float st = cap > 0.f ? cap * tanh_fast(xt * icap) : xt;
      out += rw[(long)k * rows + row] * (l - (1.0f - eps) * st - eps * mean_s);
    }
    loss[row] = out;
  }
}

template <typename IDX>
__global__ __launch_bounds__(256) void loss_multi_bwd_kernel(const bf16_t* __restrict__ x, const IDX* __restrict__ tg,
                                                            const float* __restrict__ rw, int K, long rows,
                                                            const float* __restrict__ lse, const float* __restrict__ g,
                                                            bf16_t* __restrict__ dx, int V, float cap, float eps) {
  const long row = blockIdx.x;
  const bf16_t* xr = x + row * V;
  bf16_t* dr = dx + row * V;
  long tk[LOSS_KMAX];
  float wk[LOSS_KMAX];
  float W = 0.f;
#pragma unroll
  for (int k = 0; k < LOSS_KMAX; ++k) {
    tk[k] = -1;
    wk[k] = 0.f;
    if (k < K) {
      tk[k] = (long)tg[(long)k * rows + row];
      if ((unsigned long)tk[k] < (unsigned long)V) {
        wk[k] = rw[(long)k * rows + row];
        W += wk[k];
      }
    }
  }
  const float gr = g[row];
  const float l = lse[row];
  const float icap = cap > 0.f ? 1.0f / cap : 0.f;
  const float flat = W * eps / (float)V, keep = 1.0f - eps;
  for (int i = threadIdx.x * 8; i < V; i += 256 * 8) {
    u32x4 u = *(const u32x4*)(xr + i);
    float v[8], d[8];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      v[2 * k] = bflo(u[k]);
      v[2 * k + 1] = bfhi(u[k]);
    }
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      float hot = 0.f;
#pragma unroll
      for (int k = 0; k < LOSS_KMAX; ++k) hot += (i + e == tk[k]) ? wk[k] : 0.f;
      if (cap > 0.f) {
        const float t = tanh_fast(v[e] * icap);
        d[e] = gr * (W * fexp(cap * t - l) - keep * hot - flat) * (1.0f - t * t);
      } else {
        d[e] = gr * (W * fexp(v[e] - l) - keep * hot - flat);
      }
    }
    u32x4 o = {pack2bf(d[0], d[1]), pack2bf(d[2], d[3]), pack2bf(d[4], d[5]), pack2bf(d[6], d[7])};
    *(u32x4*)(dr + i) = o;
  }
}

// ------------------------------------------------------------------------------------ LM head GEMM + lse partials
struct EpiLmHead {
  static constexpr bool kTileEpilogue = true;
  bf16_t* logits;  // [rows][V]
  float* part;     // [V/64][rows][2] (max, sum): slab-major, so that a wavefront's 32 rows of one slab are one 256-byte store
  long V, rows;
  int nchunk;      // V / 64
  float cap;
  template <int TP, int TQ>
  __device__ __forceinline__ void tile(const f32x16 (&acc)[TP][TQ], int pw, int qw, int lr, int lh, int, int) const {
    static_assert(TP == 2, "a wavefront spans 64 vocabulary columns");
    const float icap = cap > 0.f ? 1.0f / cap : 0.f;
#pragma unroll
    for (int j = 0; j < TQ; ++j) {
      const long row = qw + j * 32 + lr;
      float v[TP * 16];
#pragma unroll
      for (int i = 0; i < TP; ++i)
#pragma unroll
        for (int jj = 0; jj < 4; ++jj) {
          const int p = pw + i * 32 + jj * 8 + lh * 4;
          uint32_t w0 = pack2bf(acc[i][j][4 * jj], acc[i][j][4 * jj + 1]);
          uint32_t w1 = pack2bf(acc[i][j][4 * jj + 2], acc[i][j][4 * jj + 3]);
          u32x2 o = {w0, w1};
          *(u32x2*)(logits + row * V + p) = o;
          v[i * 16 + 4 * jj] = bflo(w0);
          v[i * 16 + 4 * jj + 1] = bfhi(w0);
          v[i * 16 + 4 * jj + 2] = bflo(w1);
          v[i * 16 + 4 * jj + 3] = bfhi(w1);
        }
      MS a;
      if (cap > 0.f) {
        a.m = cap;
        a.s = 0.f;
#pragma unroll
        for (int k = 0; k < TP * 16; ++k) a.s += capped_exp(v[k], icap, cap);
        a.s += __shfl_xor(a.s, 32, 64);
      } else {
        float mx = v[0];
#pragma unroll
        for (int k = 1; k < TP * 16; ++k) mx = fmaxf(mx, v[k]);
        mx = fmaxf(mx, __shfl_xor(mx, 32, 64));
        float t = 0.f;
#pragma unroll
        for (int k = 0; k < TP * 16; ++k) t += fexp(v[k] - mx);
        t += __shfl_xor(t, 32, 64);
        a.m = mx;
        a.s = t;
      }
      if (lh == 0) *(f32x2_t*)(part + ((long)(pw >> 6) * rows + row) * 2) = f32x2_t{a.m, a.s};
    }
  }
};

// A workgroup per 64 rows, a lane per row: each wavefront merges a quarter of the row's slab pairs (eight coalesced 512-byte
// loads in flight), the four quarters meet in LDS, then the target logit is read and lse and the row loss are written.
template <typename IDX>
__global__ __launch_bounds__(256) void lmhead_finish_kernel(const float* __restrict__ part, const bf16_t* __restrict__ logits,
                                                           const IDX* __restrict__ tg, const float* __restrict__ row_w,
                                                           float* __restrict__ loss, float* __restrict__ lse, long rows, long V,
                                                           int nchunk, float cap) {
  __shared__ float rm[4][64], rs[4][64];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const long row = (long)blockIdx.x * 64 + lane;
  const long rr = row < rows ? row : rows - 1;
  const int q = (nchunk + 3) / 4, c0 = wave * q, c1 = c0 + q < nchunk ? c0 + q : nchunk;
  MS a{-1e30f, 0.f};
  for (int c = c0; c < c1; c += 8) {
    f32x2_t v[8];
#pragma unroll
    for (int j = 0; j < 8; ++j)
      v[j] = c + j < c1 ? *(const f32x2_t*)(part + ((long)(c + j) * rows + rr) * 2) : f32x2_t{-1e30f, 0.f};
#pragma unroll
    for (int j = 0; j < 8; ++j) a = ms_merge(a, MS{v[j][0], v[j][1]});
  }
  rm[wave][lane] = a.m;
  rs[wave][lane] = a.s;
  __syncthreads();
  if (wave == 0 && row < rows) {
#pragma unroll
    for (int w = 1; w < 4; ++w) a = ms_merge(a, MS{rm[w][lane], rs[w][lane]});
    float l = a.m + logf(a.s);
    lse[row] = l;
    long tt = (long)tg[row];
    float out = 0.f;
    if ((unsigned long)tt < (unsigned long)V) {  // a target outside [0, V) is an ignored row, never an address
      float xt = bf2f(logits[row * V + tt]);
      float st = cap > 0.f ? cap * tanh_fast(xt / cap) : xt;
      out = (l - st) * (row_w ? row_w[row] : 1.0f);
    }
    loss[row] = out;
  }
}

}  // namespace

template <bool EVAL>
static void launch_loss_fwd(const void* logits, const void* targets, int idx64, const void* row_w, void* loss, void* lse, long rows,
                            int V, float softcap, hipStream_t s) {
#define TFB_LF(IDX, TPR)                                                                                                     \
  hipLaunchKernelGGL((loss_fwd_kernel<IDX, TPR, EVAL>), dim3((unsigned)((rows + 256 / TPR - 1) / (256 / TPR))), dim3(256), 0, s,    \
                     (const bf16_t*)logits, (const IDX*)targets, (const float*)row_w, (float*)loss, (float*)lse, rows, V, softcap)
  if (V <= WAVE_ROW_V) {
    if (idx64) TFB_LF(long, 64); else TFB_LF(int, 64);
  } else {
    if (idx64) TFB_LF(long, 256); else TFB_LF(int, 256);
  }
#undef TFB_LF
}

// logits bf16 [rows][V]; targets int64 (idx64) or int32, negative = ignored; row_w fp32 [rows] or NULL;
// loss fp32 [rows] (already weighted); lse fp32 [rows]. softcap <= 0 means no softcap.
extern "C" int tfb_loss_fwd(const void* logits, const void* targets, int idx64, const void* row_w, void* loss, void* lse,
                            long rows, int V, float softcap, void* stream) {
  if (!logits || !targets || !loss || !lse) return TFB_ERR_ARG;
  if (rows <= 0 || V <= 0 || V % 8) return TFB_ERR_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  launch_loss_fwd<false>(logits, targets, idx64, row_w, loss, lse, rows, V, softcap, s);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}

// w fp32 [rows]: the weight of each row's loss in the reduction, valid / max(1, number of valid rows) for the mean over the
// rows that count (mean != 0: F.cross_entropy(ignore_index < 0) semantics), valid for the sum; valid = 0 <= t < V, the rows
// the loss kernels give a loss to (V <= 0: no upper bound). One small launch in place of a compare, a cast, a sum, a clamp
// and a division.
extern "C" int tfb_loss_row_weights(const void* targets, int idx64, void* w, long rows, int mean, int V, void* stream) {
  if (!targets || !w) return TFB_ERR_ARG;
  if (rows <= 0) return TFB_ERR_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  const long vmax = V > 0 ? (long)V : (1L << 62);
  if (idx64)
    hipLaunchKernelGGL(loss_row_weights_kernel<long>, dim3(1), dim3(1024), 0, s, (const long*)targets, (float*)w, rows, mean, vmax);
  else
    hipLaunchKernelGGL(loss_row_weights_kernel<int>, dim3(1), dim3(1024), 0, s, (const int*)targets, (float*)w, rows, mean, vmax);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}

// tfb_loss_fwd followed by tfb_loss_bwd with grow = row_w (an upstream gradient of one), in place and in one pass over the
// logits: loss and lse as tfb_loss_fwd writes them, and logits overwritten by that gradient, bit for bit what the two calls
// give. V <= 65536 (a row is held in one workgroup's registers); status TFB_ERR_SHAPE beyond, for the caller to take the two calls.
extern "C" int tfb_loss_fwd_bwd(void* logits, const void* targets, int idx64, const void* row_w, void* loss, void* lse, long rows,
                                int V, float softcap, void* stream) {
  if (!logits || !targets || !loss || !lse) return TFB_ERR_ARG;
  if (rows <= 0 || V <= 0 || V % 8 || V > 65536) return TFB_ERR_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  const long blocks = V <= WAVE_ROW_V ? (rows + 3) / 4 : rows;
  const bool each = loss_each(blocks, softcap);
#define TFB_LFB(NCH, TPR, EACH, TWICE)                                                                                         \
  do {                                                                                                                         \
    if (idx64) hipLaunchKernelGGL((loss_fwd_bwd_kernel<long, NCH, TPR, EACH, TWICE>), dim3((unsigned)blocks), dim3(256), 0, s, (bf16_t*)logits,  \
                                  (const long*)targets, (const float*)row_w, (float*)loss, (float*)lse, rows, V, softcap);     \
    else hipLaunchKernelGGL((loss_fwd_bwd_kernel<int, NCH, TPR, EACH, TWICE>), dim3((unsigned)blocks), dim3(256), 0, s, (bf16_t*)logits,         \
                            (const int*)targets, (const float*)row_w, (float*)loss, (float*)lse, rows, V, softcap);            \
  } while (0)
  if (V > 32768) {
    TFB_LFB(32, 256, false, true);
  } else if (V > 16384) {
    if (softcap > 0.f) TFB_LFB(16, 256, false, true); else TFB_LFB(16, 256, false, false);
  } else if (V > 8192) {
    if (each) TFB_LFB(8, 256, true, false); else TFB_LFB(8, 256, false, false);
  } else if (V > WAVE_ROW_V) {
    if (each) TFB_LFB(4, 256, true, false); else TFB_LFB(4, 256, false, false);
  } else {
    if (each) TFB_LFB(4, 64, true, false); else TFB_LFB(4, 64, false, false);
  }
#undef TFB_LFB
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}

// dlogits may alias logits (in place). grow fp32 [rows] = upstream gradient of each row's loss times its weight.
extern "C" int tfb_loss_bwd(const void* logits, const void* targets, int idx64, const void* lse, const void* grow, void* dlogits,
                            long rows, int V, float softcap, void* stream) {
  if (!logits || !targets || !lse || !grow || !dlogits) return TFB_ERR_ARG;
  if (rows <= 0 || V <= 0 || V % 8) return TFB_ERR_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  const long blocks = V <= WAVE_ROW_V ? (rows + 3) / 4 : rows;
  const bool each = loss_each(blocks, softcap);
#define TFB_LB(TPR, EACH)                                                                                                      \
  do {                                                                                                                         \
    if (idx64) hipLaunchKernelGGL((loss_bwd_kernel<long, TPR, EACH>), dim3((unsigned)blocks), dim3(256), 0, s, (const bf16_t*)logits,  \
                                  (const long*)targets, (const float*)lse, (const float*)grow, (bf16_t*)dlogits, rows, V, softcap);    \
    else hipLaunchKernelGGL((loss_bwd_kernel<int, TPR, EACH>), dim3((unsigned)blocks), dim3(256), 0, s, (const bf16_t*)logits,         \
                            (const int*)targets, (const float*)lse, (const float*)grow, (bf16_t*)dlogits, rows, V, softcap);           \
  } while (0)
  if (V <= WAVE_ROW_V) {
    if (each) TFB_LB(64, true); else TFB_LB(64, false);
  } else {
    if (each) TFB_LB(256, true); else TFB_LB(256, false);
  }
#undef TFB_LB
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}

// Several targets per row and / or label smoothing: targets [K][rows], row_w fp32 [K][rows], 1 <= K <= 8, 0 <= eps < 1.
extern "C" int tfb_loss_multi_fwd(const void* logits, const void* targets, int idx64, const void* row_w, int K, float eps,
                                  void* loss, void* lse, long rows, int V, float softcap, void* stream) {
  if (!logits || !targets || !row_w || !loss || !lse) return TFB_ERR_ARG;
  if (rows <= 0 || V <= 0 || V % 8 || K < 1 || K > LOSS_KMAX || !(eps >= 0.f && eps < 1.f)) return TFB_ERR_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  if (idx64)
    hipLaunchKernelGGL(loss_multi_fwd_kernel<long>, dim3((unsigned)rows), dim3(256), 0, s, (const bf16_t*)logits,
                       (const long*)targets, (const float*)row_w, K, rows, (float*)loss, (float*)lse, V, softcap, eps);
  else
    hipLaunchKernelGGL(loss_multi_fwd_kernel<int>, dim3((unsigned)rows), dim3(256), 0, s, (const bf16_t*)logits,
                       (const int*)targets, (const float*)row_w, K, rows, (float*)loss, (float*)lse, V, softcap, eps);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}

// g fp32 [rows] = upstream gradient of each row's loss (the weights are applied here). dlogits may alias logits.
extern "C" int tfb_loss_multi_bwd(const void* logits, const void* targets, int idx64, const void* row_w, int K, float eps,
                                  const void* lse, const void* g, void* dlogits, long rows, int V, float softcap, void* stream) {
  if (!logits || !targets || !row_w || !lse || !g || !dlogits) return TFB_ERR_ARG;
  if (rows <= 0 || V <= 0 || V % 8 || K < 1 || K > LOSS_KMAX || !(eps >= 0.f && eps < 1.f)) return TFB_ERR_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  if (idx64)
    hipLaunchKernelGGL(loss_multi_bwd_kernel<long>, dim3((unsigned)rows), dim3(256), 0, s, (const bf16_t*)logits,
                       (const long*)targets, (const float*)row_w, K, rows, (const float*)lse, (const float*)g,
                       (bf16_t*)dlogits, V, softcap, eps);
  else
    hipLaunchKernelGGL(loss_multi_bwd_kernel<int>, dim3((unsigned)rows), dim3(256), 0, s, (const bf16_t*)logits,
                       (const int*)targets, (const float*)row_w, K, rows, (const float*)lse, (const float*)g,
                       (bf16_t*)dlogits, V, softcap, eps);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}

// Fused LM head forward: x bf16 [rows][d], W bf16 [V][d] -> logits bf16 [rows][V], loss fp32 [rows], lse fp32 [rows].
// part: fp32 scratch [rows][V/64][2].
extern "C" int tfb_lmhead_fwd(const void* x, const void* W, const void* targets, int idx64, const void* row_w, void* logits,
                              void* part, void* loss, void* lse, long rows, int d, int V, float softcap, void* stream) {
  if (!x || !W || !targets || !logits || !part || !loss || !lse) return TFB_ERR_ARG;
  if (rows <= 0 || rows % 128 || V <= 0 || V % 128 || d <= 0 || d % 64) return TFB_ERR_SHAPE;
  hipStream_t s = (hipStream_t)stream;
  // 128 x 128 tiles, two workgroups per CU started half a tile apart (gemm_core.hpp): the epilogue of one (2.1 GB of
  // logits written, exp / max / sum per element) runs under the other's MFMAs. Measured at V = 32768, 32768 rows:
  // 2.08 ms, against 2.26 ms for 256 x 256 tiles on 8 wavefronts (half the operand bytes per flop, but one resident
  // workgroup and nothing to hide its epilogue behind); a wavefront spans 64 vocabulary columns.
  using Cfg = GemmCfg<128, 128, 2, 2, 2, TFB_K_CONTIG, TFB_K_CONTIG>;
  GemmOperand P{(const uint8_t*)W, (long)d * 2}, Q{(const uint8_t*)x, (long)d * 2};
  int st;
  // Where the persistent 256 x 256 kernel takes the shape, its plain store and a pass over the logits are cheaper than the
  // exponentials in an epilogue that nothing overlaps (the call, without / with a softcap: 9600 x 8192 x 1024 261 -> 204 us /
  // 264 -> 201, 2048 x 32768 x 768 150 -> 120 / 161 -> 138, 32768 x 32768 x 768 2166 -> 2005 / 2292 -> 2199).
  if (gemm_pp_try<2, TFB_K_CONTIG, TFB_K_CONTIG, 0, 0>(P, Q, V, (int)rows, (long)d * 2, false, EpiStore{logits, (long)V, 0, 0}, s, st)) {
    if (st != TFB_OK) return st;
    launch_loss_fwd<true>(logits, targets, idx64, row_w, loss, lse, rows, V, softcap, s);
    TFB_LAUNCH_CHECK();
    return TFB_OK;
  }
  EpiLmHead e{(bf16_t*)logits, (float*)part, (long)V, rows, V / 64, softcap};
  if (!gemm_ring_try<2, TFB_K_CONTIG, TFB_K_CONTIG, 0, 0>(P, Q, V, (int)rows, (long)d * 2, e, s, st))
    st = gemm_launch<Cfg>(P, Q, V, (int)rows, (long)d * 2, 1, LoadIdentity{}, LoadIdentity{}, e, s);
  if (st != TFB_OK) return st;
  unsigned nb = (unsigned)((rows + 63) / 64);
  if (idx64)
    hipLaunchKernelGGL(lmhead_finish_kernel<long>, dim3(nb), dim3(256), 0, s, (const float*)part, (const bf16_t*)logits,
                       (const long*)targets, (const float*)row_w, (float*)loss, (float*)lse, rows, (long)V, V / 64, softcap);
  else
    hipLaunchKernelGGL(lmhead_finish_kernel<int>, dim3(nb), dim3(256), 0, s, (const float*)part, (const bf16_t*)logits,
                       (const int*)targets, (const float*)row_w, (float*)loss, (float*)lse, rows, (long)V, V / 64, softcap);
  TFB_LAUNCH_CHECK();
  return TFB_OK;
}
