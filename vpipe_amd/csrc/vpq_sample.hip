// Stochastic tail of a decode step: the full sampler over one row of logits, on the device, so that the
// drawn token never leaves it (gpu-kernels/metal/ops/llm_elementwise.metal:3063-3298, `sample_topp_f16`).
// One workgroup.  The pipeline and its order are the reference's:
//   repetition penalty -> presence penalty -> temperature -> softmax weights -> top-k -> min-p -> top-p
//   -> multinomial draw by the Gumbel-max trick,
// with the three filters as weight thresholds (no sort of the vocabulary):
//   eff_i  = seen[i] ? (v >= 0 ? v / rep : v * rep) - pres : v                         (:3106-3113)
//   w_i    = exp((eff_i - max eff) / temp), cached in `ws` in the element type; Z = sum of the w_i (fp32, unrounded)
//   t_k    = largest t of a bisection of [0, 1] with count{ws_i >= t} >= top_k           (:3170-3193; 0 < top_k < V)
//   floor  = max(t_k, min_p)   (the largest weight is 1, so min-p's probability floor is a weight floor)
//   wt     = largest t of a bisection of [floor, 1] with sum{ws_i : ws_i >= t} >= top_p Z (:3203-3222)
//   pick   = argmax over {ws_i >= wt} of eff_i / temp - log(-log(u_i)), u_i a hash of (seed, i), lowest index on
//            ties; 0 if nothing is kept; seen[pick] = 1                                   (:3224-3262)
//
// What is fixed here beyond the reference (Metal's fast math and reduction order are not defined to the bit): every
// floating-point step is written so that a plain C restatement gives the same bits -- exp and log are polynomials
// over explicit fp32 multiplies and adds (no contraction into fma in this file), a thread takes the indices
// t, t + 1024, ... in ascending order and the 1024 partial results meet in a halving tree
// (a[t] op= a[t + s], s = 512 .. 1), the reference's own pattern.  The draw is therefore an exact function of
// (logits, seen, parameters, seed), checked as index work, not to a tolerance.
#include "vpq_device.h"
#include "vpq_internal.h"

#pragma clang fp contract(off)

namespace vpq {

namespace {

constexpr int kSampleThreads = 1024;

// exp(x) for x <= 0: 2^n * p(r), n = rint(x log2 e), r = x - n ln 2 in two pieces, p the degree-5 polynomial of
// the Cephes expf.  Below -87 the result is 0.
__device__ __forceinline__ float sample_exp(float x)
{
  if (!(x >= -87.0f)) { return 0.0f; }
  const float n = __builtin_rintf(x * 1.44269504088896341f);
  float r = x - n * 0.693359375f;
  r = r - n * -2.12194440e-4f;
  float p = 1.9875691500e-4f;
  p = p * r + 1.3981999507e-3f;
  p = p * r + 8.3334519073e-3f;
  p = p * r + 4.1665795894e-2f;
  p = p * r + 1.6666665459e-1f;
  p = p * r + 5.0000001201e-1f;
  p = p * (r * r) + r;
  p = p + 1.0f;
  return p * __uint_as_float((uint32_t)((int)n + 127) << 23);
}

// log(x) for normal x > 0 (the Cephes logf): x = m 2^e with m in [sqrt(1/2), sqrt(2)), a degree-8 polynomial in
// m - 1, e ln 2 added in two pieces.
__device__ __forceinline__ float sample_log(float x)
{
  const uint32_t bits = __float_as_uint(x);
  int e = (int)(bits >> 23) - 126;
  float m = __uint_as_float((bits & 0x007fffffu) | 0x3f000000u);      // [0.5, 1)
  if (m < 0.707106781186547524f) {
    e -= 1;
    m = m + m - 1.0f;
  } else {
    m = m - 1.0f;
  }
  const float z = m * m;
  float y = 7.0376836292e-2f;
  y = y * m + -1.1514610310e-1f;
  y = y * m + 1.1676998740e-1f;
  y = y * m + -1.2420140846e-1f;
  y = y * m + 1.4249322787e-1f;
  y = y * m + -1.6668057665e-1f;
  y = y * m + 2.0000714765e-1f;
  y = y * m + -2.4999993993e-1f;
  y = y * m + 3.3333331174e-1f;
  y = y * m * z;
  const float fe = (float)e;
  y = y + fe * -2.12194440e-4f;
  y = y - 0.5f * z;
  float r = m + y;
  r = r + fe * 0.693359375f;
  return r;
}

// (llm_elementwise.metal:3096-3104) bias-reduced integer hash -> uniform in (0, 1]
__device__ __forceinline__ float sample_hash_u01(uint32_t x)
{
  x ^= x >> 16; x *= 0x7feb352dU;
  x ^= x >> 15; x *= 0x846ca68bU;
  x ^= x >> 16;
  return ((float)x + 0.5f) * (1.0f / 4294967296.0f);
}

__device__ __forceinline__ float sample_eff(float v, bool seen, float rep, float pres)
{
  if (seen) {
    v = (v >= 0.0f) ? (v / rep) : (v * rep);
    v -= pres;
  }
  return v;
}

template <typename T, typename Op>
__device__ __forceinline__ T tree(T* a, T mine, Op op)
{
  const int t = threadIdx.x;
  a[t] = mine;
  __syncthreads();
  for (int s = kSampleThreads >> 1; s > 0; s >>= 1) {
    if (t < s) { a[t] = op(a[t], a[t + s]); }
    __syncthreads();
  }
  const T r = a[0];
  __syncthreads();
  return r;
}

__global__ __launch_bounds__(kSampleThreads) void sample_topp_kernel(
    const uint16_t* __restrict__ logits, int32_t* __restrict__ out_id, int V, float temp, float top_p, uint32_t seed,
    uint16_t* __restrict__ ws, int n_iter, float rep, float pres, int top_k, float min_p, uint8_t* __restrict__ seen)
{
  __shared__ float tg[kSampleThreads];
  __shared__ int tgi[kSampleThreads];
  const int t = threadIdx.x;
  const float inv_t = 1.0f / fmaxf(temp, 1e-6f);
  auto fmax_op = [](float a, float b) { return a > b ? a : b; };     // a NaN on the right is never taken
  auto fadd_op = [](float a, float b) { return a + b; };
  auto iadd_op = [](int a, int b) { return a + b; };

  // 1) the largest penalised logit
  float m = -INFINITY;
  for (int i = t; i < V; i += kSampleThreads) {
    const float e = sample_eff(bf16_bits_to_f32(logits[i]), seen[i] != 0, rep, pres);
    m = e > m ? e : m;
  }
  const float maxl = tree(tg, m, fmax_op);

  // 2) the weights, cached in the element type, and their sum
  float z = 0.0f;
  for (int i = t; i < V; i += kSampleThreads) {
    const float e = sample_eff(bf16_bits_to_f32(logits[i]), seen[i] != 0, rep, pres);
    const float w = sample_exp((e - maxl) * inv_t);
    ws[i] = (uint16_t)f32_to_bf16_bits(w);
    z = z + w;
  }
  __threadfence_block();
  const float Z = tree(tg, z, fadd_op);
  const float target = top_p * Z;

  // 3a) top-k as a weight threshold
  float t_k = 0.0f;
  if (top_k > 0 && top_k < V) {
    float lo = 0.0f, hi = 1.0f;
    for (int it = 0; it < n_iter; ++it) {
      const float mid = 0.5f * (lo + hi);
      int cnt = 0;
      for (int i = t; i < V; i += kSampleThreads) {
        if (bf16_bits_to_f32(ws[i]) >= mid) { ++cnt; }
      }
      const int C = tree(tgi, cnt, iadd_op);
      if (C >= top_k) { lo = mid; } else { hi = mid; }
    }
    t_k = lo;
  }
  // 3b) min-p as a weight floor
  const float t_mp = fmaxf(min_p, 0.0f);
  const float t_floor = fmaxf(t_k, t_mp);

  // 3c) the nucleus threshold over the survivors
  float lo = t_floor, hi = 1.0f;
  for (int it = 0; it < n_iter; ++it) {
    const float mid = 0.5f * (lo + hi);
    float mass = 0.0f;
    for (int i = t; i < V; i += kSampleThreads) {
      const float w = bf16_bits_to_f32(ws[i]);
      if (w >= mid) { mass = mass + w; }
    }
    const float M = tree(tg, mass, fadd_op);
    if (M >= target) { lo = mid; } else { hi = mid; }
  }
  const float wt = fmaxf(lo, t_floor);

  // 4) Gumbel-max over the kept set, lowest index on ties
  float best = -INFINITY;
  int bi = -1;
  for (int i = t; i < V; i += kSampleThreads) {
    if (bf16_bits_to_f32(ws[i]) >= wt) {
      const float e = sample_eff(bf16_bits_to_f32(logits[i]), seen[i] != 0, rep, pres);
      const float u = sample_hash_u01(seed ^ ((uint32_t)i * 2654435761u + 1u));
      const float a = 0.0f - sample_log(u + 1e-20f) + 1e-20f;
      const float g = 0.0f - sample_log(a);
      const float score = e * inv_t + g;
      if (score > best) { best = score; bi = i; }
    }
  }
  tg[t] = best;
  tgi[t] = bi;
  __syncthreads();
  for (int s = kSampleThreads >> 1; s > 0; s >>= 1) {
    if (t < s) {
      const bool take = tg[t + s] > tg[t] || (tg[t + s] == tg[t] && tgi[t + s] >= 0 && (tgi[t] < 0 || tgi[t + s] < tgi[t]));
      if (take) { tg[t] = tg[t + s]; tgi[t] = tgi[t + s]; }
    }
    __syncthreads();
  }
  if (t == 0) {
    const int pick = tgi[0] >= 0 ? tgi[0] : 0;
    out_id[0] = pick;
    seen[pick] = 1;
  }
}

// ---- the sampler over many workgroups, thresholds from a histogram ----------------------------------------------
// (llm_elementwise.metal:3255-3640: `sample_max_partial_f16`, `sample_max_combine_f16`, `sample_zhist_partial_f16`,
// `sample_zhist_combine_f16`, `sample_thresh_f16`, `sample_pick_partial_f16`, `sample_pick_combine_f16`.)  The
// vocabulary is cut into n_slabs contiguous slabs, one workgroup each; top-k and top-p become the low
// edge of a histogram bin (1024 bins uniform in -log w over [0, 40), bin 0 the largest weights), so the kept set is
// the exact sampler's plus at most one bin's worth of weights.  Four launches instead of the reference's seven: the
// combine of the maxima is the prologue of the weight pass (every workgroup reduces the n_slabs maxima itself),
// the combine of the histograms and the threshold scan are one workgroup, and the draw's last workgroup stores the token.
//   work (fp32 words): [0, S) slab maxima | S x (2 B + 1): per slab counts, masses, Z | 2 B + 1: the draw's best
//   entry and its count of workgroups | 1: the weight threshold | 2 S: unused
// Exactness as above: Z of a slab is the sum of 256 partial ones, the t-th over lo + t, lo + t + 256, ... in ascending
// order, that meet in a halving tree; slabs are added in slab order; counts and the fixed-point masses of a slab are
// integer sums; a maximum does not depend on its order.
// Bound by launches and the latency of each one's loads (a slab is about 4000 entries): 1024 threads, four entries of
// each in flight, and few LDS atomics on one bin.  Measured (us at 151936 entries, 256 threads that took one after the other
// and a launch for the combine of the draw; now): maxima 9.3, weights 10.4, threshold 7.4, draw 8.2 + 4.0 -> 4.9, 5.2 (9.7 with
// two LDS atomics an entry), 5.2, 4.5.
constexpr int kHistThreads = 1024;
constexpr int kHistWaves = kHistThreads / kWave;
constexpr int kHistBatch = 4;                       // entries of a thread in flight
constexpr int kHistStep = kHistBatch * kHistThreads;
constexpr int kHistBins = 1024;
constexpr float kHistBinWidth = 40.0f / 1024.0f;
constexpr int kHistChunk = kHistThreads / 2;        // bins whose counts and masses one pass of the threshold scan adds up
constexpr int kHistSlabs = 32;                      // slabs that it has in flight

__device__ __forceinline__ int sample_bin(float w)
{
  const float lw = 0.0f - sample_log(w > 1e-30f ? w : 1e-30f);
  int b = (int)(lw / kHistBinWidth);
  if (b < 0) { b = 0; }
  if (b >= kHistBins) { b = kHistBins - 1; }
  return b;
}

// The largest value of the workgroup, in every thread (no NaN comes in).
__device__ __forceinline__ float hist_max(float* red, float m)
{
#pragma unroll
  for (int off = kWave / 2; off >= 1; off >>= 1) {
    const float o = __shfl_xor(m, off, kWave);
    m = o > m ? o : m;
  }
  if ((threadIdx.x & 63) == 0) { red[threadIdx.x >> 6] = m; }
  __syncthreads();
  m = red[0];
#pragma unroll
  for (int k = 1; k < kHistWaves; ++k) { m = red[k] > m ? red[k] : m; }
  return m;
}

// A thread's entries of the batch from i0 on: i0 + t + 1024 j; past the slab's end its last one again.
struct HistEntries {
  float v[kHistBatch];
  bool seen[kHistBatch];
};
__device__ __forceinline__ HistEntries hist_entries(const uint16_t* logits, const uint8_t* seen, int i0, int hi)
{
  HistEntries r;
#pragma unroll
  for (int j = 0; j < kHistBatch; ++j) {
    const int i = i0 + (int)threadIdx.x + j * kHistThreads, at = i < hi ? i : hi - 1;
    r.v[j] = bf16_bits_to_f32(logits[at]);
    r.seen[j] = seen[at] != 0;
  }
  return r;
}

__global__ __launch_bounds__(kHistThreads) void sample_hist_max_kernel(
    const uint16_t* __restrict__ logits, float* __restrict__ slab_max, int V, int slab, float rep, float pres,
    const uint8_t* __restrict__ seen)
{
  __shared__ float red[kHistWaves];
  const int lo = blockIdx.x * slab;
  const int hi = lo + slab < V ? lo + slab : V;
  float m = -INFINITY;
  for (int i0 = lo; i0 < hi; i0 += kHistStep) {
    const HistEntries x = hist_entries(logits, seen, i0, hi);
#pragma unroll
    for (int j = 0; j < kHistBatch; ++j) {
      const float e = sample_eff(x.v[j], x.seen[j], rep, pres);
      m = e > m ? e : m;
    }
  }
  const float r = hist_max(red, m);
  if (threadIdx.x == 0) { slab_max[blockIdx.x] = r; }
}

__global__ __launch_bounds__(kHistThreads) void sample_hist_weights_kernel(
    const uint16_t* __restrict__ logits, uint16_t* __restrict__ ws, const float* __restrict__ slab_max,
    float* __restrict__ partials, int V, int slab, int n_slabs, float temp, float rep, float pres,
    const uint8_t* __restrict__ seen)
{
  __shared__ float red[kHistWaves];
  __shared__ float batch[kHistStep];
  __shared__ uint32_t h_cnt[kHistBins];
  __shared__ uint32_t h_mass[kHistBins];
  static_assert(kHistBins == kHistThreads, "a thread has one bin");
  const int t = threadIdx.x;
  const int lo = blockIdx.x * slab;
  const int hi = lo + slab < V ? lo + slab : V;
  HistEntries x{};
  if (lo < hi) { x = hist_entries(logits, seen, lo, hi); }        // (on their way while the maxima meet)
  float m = -INFINITY;
  for (int p = t; p < n_slabs; p += kHistThreads) { m = slab_max[p] > m ? slab_max[p] : m; }
  h_cnt[t] = 0u;
  h_mass[t] = 0u;
  const float maxl = hist_max(red, m);                            // (its barrier also opens the histogram)
  const float inv_t = 1.0f / fmaxf(temp, 1e-6f);
  float z = 0.0f;
  for (int i0 = lo; i0 < hi; i0 += kHistStep) {
    if (i0 > lo) { x = hist_entries(logits, seen, i0, hi); }
#pragma unroll
    for (int j = 0; j < kHistBatch; ++j) {
      const int i = i0 + t + j * kHistThreads;
      float w = 0.0f;
      bool last = false;                                          // (most of a row: counted once a wavefront)
      if (i < hi) {
        const float e = sample_eff(x.v[j], x.seen[j], rep, pres);
        w = sample_exp((e - maxl) * inv_t);
        ws[i] = (uint16_t)f32_to_bf16_bits(w);
        const int b = sample_bin(w);
        const uint32_t mass = (uint32_t)(w * 65536.0f);
        last = b == kHistBins - 1;
        if (!last) { atomicAdd(&h_cnt[b], 1u); }
        if (mass != 0) { atomicAdd(&h_mass[b], mass); }           // (none below e^-11)
      }
      const unsigned long long lasts = __ballot(last);
      if (lasts != 0 && (t & 63) == 0) { atomicAdd(&h_cnt[kHistBins - 1], (uint32_t)__builtin_popcountll(lasts)); }
      batch[t + j * kHistThreads] = w;
    }
    __syncthreads();
    if (t < 256) {
#pragma unroll
      for (int q = 0; q < kHistStep / 256; ++q) { z = z + batch[t + q * 256]; }   // (+0 past the slab's end)
    }
    __syncthreads();
  }
  if (t < 256) { batch[t] = z; }
  __syncthreads();
  float* P = partials + (size_t)blockIdx.x * (size_t)(2 * kHistBins + 1);
  P[t] = (float)h_cnt[t];
  P[kHistBins + t] = (float)h_mass[t] * (1.0f / 65536.0f);
  if (t < kWave) {                                                // a[t] += a[t + s], s = 128 .. 1
    float a = (batch[t] + batch[t + 128]) + (batch[t + 64] + batch[t + 192]);
#pragma unroll
    for (int s = kWave / 2; s >= 1; s >>= 1) { a = a + __shfl_down(a, s, kWave); }
    if (t == 0) { P[2 * kHistBins] = a; }
  }
}

// What the draw's workgroups share, in the words between the slabs' sums and the threshold: the best entry so far (the
// score as an ordered number above the complement of the index, 0: none) and how many workgroups have given theirs.
struct HistDraw {
  unsigned long long best;
  unsigned count;
};
__host__ __device__ __forceinline__ HistDraw* hist_draw(float* hist)
{
  return reinterpret_cast<HistDraw*>((reinterpret_cast<uintptr_t>(hist) + 7) & ~(uintptr_t)7);
}

// One workgroup: the slabs' histograms and Z added in slab order (a thread owns a cell of 512 bins' counts and masses; its
// loads are issued 32 at a time, the additions stay in slab order), then the reference's scan
// (gpu-kernels/metal/ops/llm_elementwise.metal:3476-3497): one thread walks the bins from 0 with one running count
// and one running mass -- the same additions in the same order, so that a crossing at a knife edge falls into the
// same bin -- and stops at the bin where both targets are met.  The upper half of the bins (weights below e^-20) is added up
// only where the walk gets there.
__global__ __launch_bounds__(kHistThreads) void sample_hist_thresh_kernel(
    const float* __restrict__ partials, float* __restrict__ hist, float* __restrict__ wt_out, int n_slabs, int V,
    float top_p, int top_k, float min_p)
{
  __shared__ __attribute__((aligned(16))) float cells[kHistThreads];   // counts of the chunk's bins, then their masses
  __shared__ float zs[kHistThreads];
  __shared__ int done_all;
  constexpr int stride = 2 * kHistBins + 1;
  const int t = threadIdx.x;
  if (t == 0) {
    HistDraw* d = hist_draw(hist);
    d->best = 0;
    d->count = 0;
  }
  float Z = 0.0f;                                     // (thread 0's)
  const bool do_k = top_k > 0 && top_k < V;
  float t_k = 0.0f, t_p = 0.0f, cum_cnt = 0.0f, cum_mass = 0.0f;
  bool have_k = false, have_p = false;
  for (int bin0 = 0; bin0 < kHistBins; bin0 += kHistChunk) {
    const int c = t < kHistChunk ? bin0 + t : kHistBins + bin0 + t - kHistChunk;
    const float zmine = bin0 == 0 && t < n_slabs ? partials[(size_t)t * stride + 2 * kHistBins] : 0.0f;
    float acc = 0.0f;
    for (int p0 = 0; p0 < n_slabs; p0 += kHistSlabs) {
      float v[kHistSlabs];
#pragma unroll
      for (int q = 0; q < kHistSlabs; ++q) {
        v[q] = partials[(size_t)(p0 + q < n_slabs ? p0 + q : n_slabs - 1) * stride + c];
      }
#pragma unroll
      for (int q = 0; q < kHistSlabs; ++q) {
        if (p0 + q < n_slabs) { acc = acc + v[q]; }
      }
    }
    cells[t] = acc;
    if (bin0 == 0) { zs[t] = zmine; }
    __syncthreads();
    if (t == 0) {
      if (bin0 == 0) {
        for (int p = 0; p < n_slabs; ++p) { Z = Z + zs[p]; }      // (1024 at most)
      }
      const float target = top_p * Z;
      bool done = false;
      for (int b0 = 0; b0 < kHistChunk && !done; b0 += 8) {
        // The sums do not fall: the eight bins hold a crossing if the last of them has crossed.
        float c8[8], m8[8];
#pragma unroll
        for (int q = 0; q < 8; ++q) {
          cum_cnt = cum_cnt + cells[b0 + q];
          cum_mass = cum_mass + cells[kHistChunk + b0 + q];
          c8[q] = cum_cnt;
          m8[q] = cum_mass;
        }
        if (do_k && !have_k && cum_cnt >= (float)top_k) {
          int q = 0;
          while (q < 7 && !(c8[q] >= (float)top_k)) { ++q; }
          t_k = sample_exp(0.0f - (float)(bin0 + b0 + q + 1) * kHistBinWidth);
          have_k = true;
        }
        if (!have_p && cum_mass >= target) {
          int q = 0;
          while (q < 7 && !(m8[q] >= target)) { ++q; }
          t_p = sample_exp(0.0f - (float)(bin0 + b0 + q + 1) * kHistBinWidth);
          have_p = true;
        }
        done = (!do_k || have_k) && have_p;
      }
      done_all = done ? 1 : 0;
    }
    __syncthreads();
    if (done_all) { break; }
  }
  if (t == 0) { wt_out[0] = fmaxf(fmaxf(t_k, fmaxf(min_p, 0.0f)), t_p); }
}

// The draw: every workgroup's best entry goes into HistDraw by one atomic maximum, whose return it waits for before it counts
// itself; so the one that finds all others counted reads the best of all.  (No data but the two atomics passes between
// workgroups: nothing to write back or to invalidate.)
__global__ __launch_bounds__(kHistThreads) void sample_hist_pick_kernel(
    const uint16_t* __restrict__ logits, const uint16_t* __restrict__ ws, const float* __restrict__ wt_in, HistDraw* draw, int V,
    int slab, float temp, uint32_t seed, float rep, float pres, uint8_t* seen, int32_t* __restrict__ out_id)
{
  __shared__ unsigned long long red[kHistWaves];
  const int t = threadIdx.x;
  const float inv_t = 1.0f / fmaxf(temp, 1e-6f);
  const float wt = wt_in[0];
  const int lo = blockIdx.x * slab;
  const int hi = lo + slab < V ? lo + slab : V;
  unsigned long long best = 0;
  for (int i0 = lo; i0 < hi; i0 += kHistStep) {
    const HistEntries x = hist_entries(logits, seen, i0, hi);
    float w[kHistBatch];
#pragma unroll
    for (int j = 0; j < kHistBatch; ++j) {
      const int i = i0 + t + j * kHistThreads;
      w[j] = bf16_bits_to_f32(ws[i < hi ? i : hi - 1]);
    }
#pragma unroll
    for (int j = 0; j < kHistBatch; ++j) {
      const int i = i0 + t + j * kHistThreads;
      if (i < hi && w[j] >= wt) {
        const float e = sample_eff(x.v[j], x.seen[j], rep, pres);
        const float u = sample_hash_u01(seed ^ ((uint32_t)i * 2654435761u + 1u));
        const float a = 0.0f - sample_log(u + 1e-20f) + 1e-20f;
        const float g = 0.0f - sample_log(a);
        const float score = e * inv_t + g + 0.0f;     // (-0 as +0: they are equal)
        if (score > -INFINITY) {
          const uint32_t bits = __float_as_uint(score), up = (bits >> 31) != 0 ? ~bits : bits | 0x80000000u;
          const unsigned long long key = (unsigned long long)up << 32 | (0xffffffffu - (uint32_t)i);
          best = key > best ? key : best;
        }
      }
    }
  }
#pragma unroll
  for (int off = kWave / 2; off >= 1; off >>= 1) {
    const unsigned long long o = __shfl_xor(best, off, kWave);
    best = o > best ? o : best;
  }
  if ((t & 63) == 0) { red[t >> 6] = best; }
  __syncthreads();                                    // (every load of `seen` has returned)
  if (t != 0) { return; }
#pragma unroll
  for (int k = 1; k < kHistWaves; ++k) { best = red[k] > best ? red[k] : best; }
  const unsigned long long before = atomicMax(&draw->best, best);
  asm volatile("s_waitcnt vmcnt(0)" : : "v"((uint32_t)before) : "memory");
  if (atomicAdd(&draw->count, 1u) != gridDim.x - 1) { return; }
  const unsigned long long key = atomicMax(&draw->best, 0ull);
  const int pick = key != 0 ? (int)(0xffffffffu - (uint32_t)key) : 0;
  out_id[0] = pick;
  seen[pick] = 1;
}

}  // namespace

size_t sample_hist_work_words(int n_slabs)
{
  return (size_t)n_slabs + (size_t)n_slabs * (2 * kHistBins + 1) + (2 * kHistBins + 1) + 1 + 2 * (size_t)n_slabs;
}

hipError_t launch_sample_hist(hipStream_t st, const uint16_t* logits, int32_t* out_id, int V, float temp, float top_p,
                              uint32_t seed, uint16_t* ws, float rep, float pres, int top_k, float min_p, uint8_t* seen,
                              int n_slabs, float* work)
{
  const int slab = (V + n_slabs - 1) / n_slabs;
  float* slab_max = work;
  float* partials = slab_max + n_slabs;
  float* hist = partials + (size_t)n_slabs * (2 * kHistBins + 1);
  float* wt = hist + (2 * kHistBins + 1);
  const dim3 slabs((unsigned)n_slabs), one(1), block(kHistThreads);
  hipError_t e = launch_kernel(sample_hist_max_kernel, slabs, block, 0, st, logits, slab_max, V, slab, rep, pres,
                               (const uint8_t*)seen);
  if (e != hipSuccess) { return e; }
  e = launch_kernel(sample_hist_weights_kernel, slabs, block, 0, st, logits, ws, (const float*)slab_max, partials, V, slab,
                    n_slabs, temp, rep, pres, (const uint8_t*)seen);
  if (e != hipSuccess) { return e; }
  e = launch_kernel(sample_hist_thresh_kernel, one, block, 0, st, (const float*)partials, hist, wt, n_slabs, V, top_p, top_k,
                    min_p);
  if (e != hipSuccess) { return e; }
  return launch_kernel(sample_hist_pick_kernel, slabs, block, 0, st, logits, (const uint16_t*)ws, (const float*)wt,
                       hist_draw(hist), V, slab, temp, seed, rep, pres, seen, out_id);
}

hipError_t launch_sample_topp(hipStream_t st, const uint16_t* logits, int32_t* out_id, int V, float temp, float top_p,
                              uint32_t seed, uint16_t* ws, int n_iter, float rep, float pres, int top_k, float min_p,
                              uint8_t* seen)
{
  return launch_kernel(sample_topp_kernel, dim3(1), dim3(kSampleThreads), 0, st, logits, out_id, V, temp, top_p, seed, ws,
                       n_iter, rep, pres, top_k, min_p, seen);
}

}  // namespace vpq
