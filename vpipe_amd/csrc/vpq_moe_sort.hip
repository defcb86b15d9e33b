// Counting sort of the (token, expert) pairs of an MoE block into per-expert blocks of slots, each
// expert's share padded to whole blocks of `block_rows` slots -- the row order the grouped expert GEMM
// multiplies in (gpu-kernels/metal/ops/llm_elementwise.metal:255-326: moe_ifill_i32, moe_hist_i32,
// moe_sort_setup_i32, moe_scatter_i32; driven by
// generative-models/qwen3/metal-qwen-model.cc:4213-4237).
//
//   tile2e[t]  expert of block t, -1 for a block no expert uses;
//   srow[i]    x (token) row of slot i = pair / top_k, -1 for a padding slot;
//   sdst[i]    the pair of slot i, -1 for a padding slot;
//   ntiles[0]  blocks in use.
// Experts come in ascending order, expert e's first slot is block_rows * (blocks of the experts below
// it).  The order of the pairs inside an expert's share is whatever order their atomic tickets come
// in; every consumer treats the slots independently, so results do not depend on it.  A pair whose
// expert id lies outside [0, n_experts) gets no slot.
//
// Up to 16384 pairs: one workgroup, one launch.  A pair's ticket is an LDS atomic, kept in a register; the slots are put
// together in LDS as 16-bit pair numbers and written out in order, 16 bytes a lane.  Bound by launch latency at few pairs and
// by one CU's LDS atomics and stores at many.  Measured against the four launches below (us, in a graph): 512 / 4096 /
// 16384 pairs of 128 experts 9.7 / 12.0 / 12.6 -> 6.4 / 7.5 / 10.7.  The line, in a kernel that takes twice as many: 16384 pairs
// of 128 / 64 / 8 experts 12.0 / 11.1 / 11.5 -> 11.5 / 10.1 / 11.3, 20480 pairs 12.0 / 11.4 / 11.7 -> 12.4 / 11.0 / 12.8.
// More pairs, or experts: four launches on the caller's stream (no allocation; ws holds 3 n_experts ints): fill, histogram,
// offsets by one wavefront (a scan over the experts), scatter.
#include <atomic>

#include "vpq_device.h"
#include "vpq_internal.h"

namespace vpq {

namespace {

__global__ __launch_bounds__(256) void moe_sort_fill_kernel(int* tile2e, int max_tiles, int* srow, int* sdst, int npad,
                                                            int* hist, int n_experts)
{
  const int stride = (int)gridDim.x * 256;
  const int cover = npad > n_experts ? npad : n_experts;     // max_tiles <= npad
  for (int i = (int)blockIdx.x * 256 + (int)threadIdx.x; i < cover; i += stride) {
    if (i < npad) {
      srow[i] = -1;
      sdst[i] = -1;
    }
    if (i < max_tiles) { tile2e[i] = -1; }
    if (i < n_experts) { hist[i] = 0; }
  }
}

// Pairs per workgroup of the histogram and scatter kernels, and the expert count up to which a workgroup
// counts in LDS first (one global atomic per expert and workgroup instead of one per pair).
constexpr int kSortChunk = 1024;
constexpr int kSortLdsExperts = 4096;

__global__ __launch_bounds__(256) void moe_sort_hist_kernel(const int* __restrict__ eid, int n_pairs, int n_experts, int* hist)
{
  __shared__ int local[kSortLdsExperts];
  const int p0 = (int)blockIdx.x * kSortChunk;
  const bool in_lds = n_experts <= kSortLdsExperts;
  if (in_lds) {
    for (int e = (int)threadIdx.x; e < n_experts; e += 256) { local[e] = 0; }
    __syncthreads();
  }
  for (int i = (int)threadIdx.x; i < kSortChunk; i += 256) {
    const int p = p0 + i;
    if (p >= n_pairs) { break; }
    const int e = eid[p];
    if (e >= 0 && e < n_experts) { atomicAdd(in_lds ? local + e : hist + e, 1); }
  }
  if (in_lds) {
    __syncthreads();
    for (int e = (int)threadIdx.x; e < n_experts; e += 256) {
      if (local[e] != 0) { atomicAdd(hist + e, local[e]); }
    }
  }
}

// One wavefront: lane l owns the experts [l * per, (l + 1) * per).
__global__ __launch_bounds__(64) void moe_sort_setup_kernel(const int* __restrict__ hist, int* boff, int* cursor, int* tile2e,
                                                            int* ntiles, int n_experts, int block_rows, int max_tiles)
{
  const int lane = (int)threadIdx.x;
  const int per = (n_experts + 63) / 64;
  const int e0 = lane * per;
  int mine = 0;                                   // blocks of this lane's experts
  for (int i = 0; i < per; ++i) {
    const int e = e0 + i;
    if (e < n_experts) { mine += (hist[e] + block_rows - 1) / block_rows; }
  }
  int incl = mine;                                // inclusive scan over the lanes
#pragma unroll
  for (int d = 1; d < 64; d <<= 1) {
    const int up = __shfl_up(incl, d, 64);
    if (lane >= d) { incl += up; }
  }
  int t = incl - mine;                            // first block of this lane's experts
  for (int i = 0; i < per; ++i) {
    const int e = e0 + i;
    if (e >= n_experts) { break; }
    const int nb = (hist[e] + block_rows - 1) / block_rows;
    boff[e] = t * block_rows;
    cursor[e] = 0;
    for (int j = 0; j < nb; ++j) {
      if (t + j < max_tiles) { tile2e[t + j] = e; }
    }
    t += nb;
  }
  if (lane == 63) { ntiles[0] = incl; }
}

__global__ __launch_bounds__(256) void moe_sort_scatter_kernel(const int* __restrict__ eid, const int* __restrict__ boff,
                                                               int* cursor, int* srow, int* sdst, int n_pairs, int top_k,
                                                               int n_experts, int npad)
{
  __shared__ int local[kSortLdsExperts];     // pairs of this workgroup per expert, then their first ticket
  const int p0 = (int)blockIdx.x * kSortChunk;
  const bool in_lds = n_experts <= kSortLdsExperts;
  int rank[kSortChunk / 256];
  if (in_lds) {
    for (int e = (int)threadIdx.x; e < n_experts; e += 256) { local[e] = 0; }
    __syncthreads();
#pragma unroll
    for (int j = 0; j < kSortChunk / 256; ++j) {
      const int p = p0 + j * 256 + (int)threadIdx.x;
      const int e = p < n_pairs ? eid[p] : -1;
      rank[j] = (e >= 0 && e < n_experts) ? atomicAdd(local + e, 1) : 0;
    }
    __syncthreads();
    for (int e = (int)threadIdx.x; e < n_experts; e += 256) {
      const int c = local[e];
      if (c != 0) { local[e] = atomicAdd(cursor + e, c); }     // a run of c tickets
    }
    __syncthreads();
  }
#pragma unroll
  for (int j = 0; j < kSortChunk / 256; ++j) {
    const int p = p0 + j * 256 + (int)threadIdx.x;
    if (p >= n_pairs) { continue; }
    const int e = eid[p];
    if (e < 0 || e >= n_experts) { continue; }
    const int ticket = in_lds ? local[e] + rank[j] : atomicAdd(cursor + e, 1);
    const int slot = boff[e] + ticket;
    if (slot < npad) {
      srow[slot] = p / top_k;
      sdst[slot] = p;
    }
  }
}

constexpr int kSortOneThreads = 1024;
constexpr int kSortOneEach = 16;                // pairs per thread, at most
constexpr int kSortOneExperts = 1024;
constexpr int kSortOneLds = 160 * 1024;

// LDS: slots [npad] of 16 bits (0xffff: padding), then per expert its count and its first slot.
__global__ __launch_bounds__(kSortOneThreads) void moe_sort_one_kernel(const int* __restrict__ eid, int n_pairs, uint32_t inv_top_k,
                                                                      int n_experts, int block_rows, int max_tiles, int* tile2e,
                                                                      int* srow, int* sdst, int* ntiles)
{
  extern __shared__ __attribute__((aligned(16))) uint16_t slots[];
  const int npad = max_tiles * block_rows, words = (npad + 7) / 8 * 4;
  uint32_t* slots2 = reinterpret_cast<uint32_t*>(slots);
  int* count = reinterpret_cast<int*>(slots2 + words);
  int* first = count + n_experts;
  int* used = first + n_experts;
  const int tid = (int)threadIdx.x;
  for (int i = tid; i < words; i += kSortOneThreads) { slots2[i] = 0xffffffffu; }
  for (int i = tid; i < n_experts; i += kSortOneThreads) { count[i] = 0; }
  int e_of[kSortOneEach];
#pragma unroll
  for (int j = 0; j < kSortOneEach; ++j) {
    const int p = j * kSortOneThreads + tid;
    e_of[j] = p < n_pairs ? eid[p] : -1;
  }
  __syncthreads();
  uint32_t ticket[kSortOneEach];                // expert in the upper half
#pragma unroll
  for (int j = 0; j < kSortOneEach; ++j) {
    ticket[j] = 0xffffffffu;
    if (j * kSortOneThreads < n_pairs && e_of[j] >= 0 && e_of[j] < n_experts) {
      ticket[j] = ((uint32_t)e_of[j] << 16) | (uint32_t)atomicAdd(count + e_of[j], 1);
    }
  }
  __syncthreads();
  if (tid < kWave) {                            // one wavefront: lane l owns the experts [l * per, (l + 1) * per)
    const int per = (n_experts + 63) / 64, e0 = tid * per;
    int mine = 0;
    for (int i = 0; i < per; ++i) {
      if (e0 + i < n_experts) { mine += (count[e0 + i] + block_rows - 1) / block_rows; }
    }
    int incl = mine;
#pragma unroll
    for (int d = 1; d < 64; d <<= 1) {
      const int up = __shfl_up(incl, d, 64);
      if (tid >= d) { incl += up; }
    }
    int t = incl - mine;
    for (int i = 0; i < per && e0 + i < n_experts; ++i) {
      const int nb = (count[e0 + i] + block_rows - 1) / block_rows;
      first[e0 + i] = t * block_rows;
      for (int j = 0; j < nb; ++j) {
        if (t + j < max_tiles) { tile2e[t + j] = e0 + i; }
      }
      t += nb;
    }
    if (tid == 63) {
      *used = incl;
      ntiles[0] = incl;
    }
  }
  __syncthreads();
#pragma unroll
  for (int j = 0; j < kSortOneEach; ++j) {
    if (j * kSortOneThreads < n_pairs && ticket[j] != 0xffffffffu) {
      const int slot = first[ticket[j] >> 16] + (int)(ticket[j] & 0xffffu);
      if (slot < npad) { slots[slot] = (uint16_t)(j * kSortOneThreads + tid); }
    }
  }
  for (int i = *used + tid; i < max_tiles; i += kSortOneThreads) { tile2e[i] = -1; }
  __syncthreads();
  // (0xffff is no pair: there are at most 16384)
  for (int i = tid * 4; i < npad; i += kSortOneThreads * 4) {
    int d[4], r[4];
#pragma unroll
    for (int k = 0; k < 4; ++k) {
      const uint32_t v = slots[i + k];          // (the array is whole eights)
      d[k] = v == 0xffffu ? -1 : (int)v;
      r[k] = v == 0xffffu ? -1 : (int)__umulhi(v, inv_top_k);
    }
    if (inv_top_k == 0u) {                      // top_k 1
#pragma unroll
      for (int k = 0; k < 4; ++k) { r[k] = d[k]; }
    }
    if (i + 3 < npad && ((reinterpret_cast<uintptr_t>(srow) | reinterpret_cast<uintptr_t>(sdst)) & 15) == 0) {
      *reinterpret_cast<int4*>(srow + i) = make_int4(r[0], r[1], r[2], r[3]);
      *reinterpret_cast<int4*>(sdst + i) = make_int4(d[0], d[1], d[2], d[3]);
    } else {
#pragma unroll
      for (int k = 0; k < 4; ++k) {
        if (i + k < npad) {
          srow[i + k] = r[k];
          sdst[i + k] = d[k];
        }
      }
    }
  }
}

// `moe_scatter_back_f16` (gpu-kernels/metal/ops/llm_elementwise.metal:328-342): rows of the sorted down
// projection back to pair order, partials[sdst[slot]] = dsorted[slot]; padding slots (sdst < 0) and destinations
// outside [0, n_pairs) are skipped.  16 bytes per thread where the rows allow, else 2.
template <typename V>
__global__ __launch_bounds__(256) void moe_scatter_back_kernel(const V* __restrict__ dsorted, const int* __restrict__ sdst,
                                                              V* __restrict__ partials, int npad, int row_vecs, int n_pairs)
{
  const size_t i = (size_t)blockIdx.x * 256 + threadIdx.x;
  if (i >= (size_t)npad * (size_t)row_vecs) { return; }
  const int slot = (int)(i / (size_t)row_vecs);
  const int v = (int)(i - (size_t)slot * (size_t)row_vecs);
  const int p = sdst[slot];
  if (p < 0 || p >= n_pairs) { return; }
  partials[(size_t)p * row_vecs + v] = dsorted[(size_t)slot * row_vecs + v];
}

}  // namespace

hipError_t launch_moe_scatter_back(hipStream_t st, const uint16_t* dsorted, const int* sdst, uint16_t* partials, int npad,
                                   int H, int n_pairs, bool wide)
{
  if (wide) {
    const size_t n = (size_t)npad * (size_t)(H / 8);
    return launch_kernel(moe_scatter_back_kernel<uint4>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st,
                         reinterpret_cast<const uint4*>(dsorted), sdst, reinterpret_cast<uint4*>(partials), npad, H / 8, n_pairs);
  }
  const size_t n = (size_t)npad * (size_t)H;
  return launch_kernel(moe_scatter_back_kernel<uint16_t>, dim3((unsigned)((n + 255) / 256)), dim3(256), 0, st, dsorted, sdst,
                       partials, npad, H, n_pairs);
}

hipError_t launch_moe_sort(hipStream_t st, const int* pair_eid, int n_pairs, int top_k, int n_experts, int block_rows,
                           int max_tiles, int* tile2e, int* srow, int* sdst, int* ntiles, int* ws)
{
  const int npad = max_tiles * block_rows;
  const size_t one_lds = (size_t)(npad + 7) / 8 * 16 + ((size_t)2 * n_experts + 1) * 4;
  if (n_pairs <= kSortOneThreads * kSortOneEach && n_experts <= kSortOneExperts && one_lds <= (size_t)kSortOneLds) {
    static std::atomic<bool> ready{false};      // (two threads may both set the attribute, which is harmless)
    if (!ready.load(std::memory_order_acquire)) {
      const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(moe_sort_one_kernel),
                                               hipFuncAttributeMaxDynamicSharedMemorySize, kSortOneLds);
      if (e != hipSuccess) { return e; }
      ready.store(true, std::memory_order_release);
    }
    // p / top_k as a multiplication by ceil(2^32 / top_k): exact for p < 2^16
    const uint32_t inv = top_k > 1 ? (uint32_t)(((1ull << 32) + (uint32_t)top_k - 1) / (uint32_t)top_k) : 0u;
    return launch_kernel(moe_sort_one_kernel, dim3(1), dim3(kSortOneThreads), one_lds, st, pair_eid, n_pairs, inv, n_experts,
                         block_rows, max_tiles, tile2e, srow, sdst, ntiles);
  }
  int* hist = ws;
  int* boff = ws + n_experts;
  int* cursor = ws + 2 * n_experts;
  const int cover = npad > n_experts ? npad : n_experts;
  int fill_blocks = (cover + 255) / 256;
  if (fill_blocks > 1024) { fill_blocks = 1024; }
  hipError_t e = launch_kernel(moe_sort_fill_kernel, dim3((unsigned)fill_blocks), dim3(256), 0, st, tile2e, max_tiles, srow,
                               sdst, npad, hist, n_experts);
  if (e != hipSuccess) { return e; }
  const dim3 pgrid((unsigned)((n_pairs + kSortChunk - 1) / kSortChunk));
  e = launch_kernel(moe_sort_hist_kernel, pgrid, dim3(256), 0, st, pair_eid, n_pairs, n_experts, hist);
  if (e != hipSuccess) { return e; }
  e = launch_kernel(moe_sort_setup_kernel, dim3(1), dim3(64), 0, st, (const int*)hist, boff, cursor, tile2e, ntiles,
                    n_experts, block_rows, max_tiles);
  if (e != hipSuccess) { return e; }
  return launch_kernel(moe_sort_scatter_kernel, pgrid, dim3(256), 0, st, pair_eid, (const int*)boff, cursor, srow, sdst,
                       n_pairs, top_k, n_experts, npad);
}

}  // namespace vpq
