// Gathered expert projections of an MoE block at decode (groups of 64, K up to 4096, 8 bits 5120): each (token, expert) pair's
// row of x against that expert's slab, one launch for all pairs (gpu-kernels/metal/quant/affine_qmv.metal:908-962, 1262-1292);
// and one row of x against up to four 8-bit packs.  Per row of weights the arithmetic and the order of every sum are those of
// the kernels of one wavefront per weight row (vpq_qmv_rows.hip, qmv_rows8_kernel), so a pair has the bits of that row's call on
// its slab.
//
// What bounds it: the slabs' read from HBM, a few megabytes a pair; the row-streaming kernel, one or two rows a wavefront,
// was bound by the vector ALU instead -- of its 140 instructions a row of 2048 values, 50 unpack and contract, the others
// order x, sum it, and reduce one row at a time over the LDS crossbar.  Here a wavefront keeps its pair's x in registers
// (32 values a lane and pass, ordered and summed once) and walks sets of weight rows, the next set's codes, scales and
// biases in flight while one is contracted; a set's row sums share their reduction: the two wide steps exchange halves
// between two rows' registers, so four rows end in the lanes of one.
// Measured (us; before: the row kernels; now), gate|up 2048 -> 2 x 768 / down 768 -> 2048 of 8 of 128 experts: 1 token 7.4 / 5.4 ->
// 6.0 / 5.0, 4 tokens 17.9 / 12.5 -> 13.5 / 9.1, 16 tokens 62 / 38 -> 37 / 23; 8 bits, 4 tokens 23.6 / 18.0 -> 21.3 / 13.1.  At 4
// tokens it reads 4.1 TB/s (8 bits 5.0), the launch's start and end included.
#include "vpq_device.h"
#include "vpq_internal.h"

namespace vpq {

namespace {

typedef __attribute__((__vector_size__(2 * sizeof(__bf16)))) __bf16 bf16x2;

__device__ __forceinline__ float gather_dot2(uint32_t a, uint32_t b, float c)
{
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2, a), __builtin_bit_cast(bf16x2, b), c, false);
}

// a's lower half-wavefront plus its upper one, in the lower lanes; b's in the upper lanes.
__device__ __forceinline__ float fold32(float a, float b)
{
  const auto r = __builtin_amdgcn_permlane32_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

// The same between neighbouring rows of 16 lanes: even rows a's sum, odd rows b's.
__device__ __forceinline__ float fold16(float a, float b)
{
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(a), __float_as_uint(b), false, false);
  return __uint_as_float(r[0]) + __uint_as_float(r[1]);
}

template <int CTRL>
__device__ __forceinline__ float add_dpp(float v)
{
  return v + __builtin_bit_cast(float, __builtin_amdgcn_update_dpp(0, __builtin_bit_cast(int, v), CTRL, 0xf, 0xf, false));
}

// Sum over the 16 lanes of a row, in every lane: steps of 8, 4, 2, 1.
__device__ __forceinline__ float row_sum(float v)
{
  v = add_dpp<0x128>(v);    // row_ror 8
  v = add_dpp<0x124>(v);    // row_ror 4 (lanes 8 apart are equal by now)
  v = add_dpp<0x4e>(v);     // quad_perm [2,3,0,1]
  return add_dpp<0xb1>(v);  // quad_perm [1,0,3,2]
}

}  // namespace

namespace {

// P: passes over K of LPR lanes by 32 values of 4 bits, 16 of 8 bits.  LPR: lanes per weight row (32: two row groups a
// wavefront, 4 bits and K up to 1024).  block, blocks: this workgroup among those of the pair, or of the pack (ONE: one row of
// x, pair_eid unread; residual and fp32 stores).
template <int BITS, int P, int LPR, bool ONE>
__device__ __forceinline__ void gather_body(const uint32_t* __restrict__ w_, const uint16_t* __restrict__ scales_,
                                            const uint16_t* __restrict__ biases_, const uint16_t* __restrict__ x_,
                                            const int* __restrict__ pair_eid, int K, int N, int x_div, int n_experts,
                                            void* __restrict__ y_, int gate_act, int block, int blocks,
                                            const uint16_t* __restrict__ residual, int y_f32)
{
  static_assert(LPR == 64 || (LPR == 32 && BITS == 4), "");
  constexpr int R = 4;                              // rows of a set and row group (the reduction below)
  constexpr int kRows = R * (kWave / LPR);          // rows of a set
  constexpr int kVals = 128 / BITS;                 // values of K per lane and pass
  constexpr int kX = kVals / 8;                     // ... of x, in 16 bytes
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int sub = lane / LPR, ll = lane % LPR;
  const int sets = (N + kRows - 1) / kRows, stride = blocks * 4;
  int set = block * 4 + wave;
  if (set >= sets) { return; }                      // (no barrier in this kernel)

  const int p = ONE ? 0 : (int)blockIdx.y;
  const uint16_t* x = x_ + (size_t)(p / x_div) * K;
  const int Kw = K * BITS / 32, Kg = K >> 6;
  // (lanes past K, which contract nothing, take the row's start: under a condition a load waited for the one before it, 4 tokens
  // of 8 of 128 experts 25.9 -> 25.0 us a layer)
  uint4 xd[P][kX];
#pragma unroll
  for (int c = 0; c < P; ++c) {
    const int k = (c * LPR + ll) * kVals, k0 = k < K ? k : 0;
#pragma unroll
    for (int t = 0; t < kX; ++t) { xd[c][t] = *reinterpret_cast<const uint4*>(x + k0 + 8 * t); }
  }
  int e = ONE ? 0 : pair_eid[p];
  const bool expert_ok = ONE || (e >= 0 && e < n_experts);
  e = expert_ok ? e : 0;
  const uint32_t* w = w_ + (size_t)e * (size_t)N * Kw;
  const uint16_t* scales = scales_ + (size_t)e * (size_t)N * Kg;
  const uint16_t* biases = biases_ + (size_t)e * (size_t)N * Kg;
  uint16_t* y = static_cast<uint16_t*>(y_) + (size_t)p * (size_t)(gate_act ? (N >> 1) : N);

  struct Pass {
    uint4 c[R];
    uint32_t s[R], b[R];
  };
  auto fetch = [&](int at, int c, Pass& v) {
    const int n0 = at * kRows + sub * R;
    const int k = (c * LPR + ll) * kVals, k0 = k < K ? k : 0;        // (lanes past K: unused)
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const int n = n0 + r < N ? n0 + r : N - 1;                     // rows past N redo the last one; never stored
      v.c[r] = *reinterpret_cast<const uint4*>(w + (size_t)n * Kw + k0 * BITS / 32);
      v.s[r] = scales[(size_t)n * Kg + (k0 >> 6)];
      v.b[r] = biases[(size_t)n * Kg + (k0 >> 6)];
    }
  };
  // The passes of a set whose loads are in flight while the set before is contracted: all, or one, as registers allow.
  constexpr int kAhead = BITS == 4 || P <= 2 ? P : 1;
  Pass cur[kAhead];
#pragma unroll
  for (int c = 0; c < kAhead; ++c) { fetch(set, c, cur[c]); }

  // 4 bits: x as pairs (x_i, x_{i+4}) of each eight values, and its sum
  uint32_t magic = 0x43004300u;                     // bf16 128.0 in both halves
  uint32_t mask = 0x000f000fu;
  asm volatile("" : "+v"(magic));                   // no instruction: hides the constants from folding, so
  asm volatile("" : "+s"(mask));                    // that each pair costs one v_and_or_b32
  const uint32_t ones = 0x3f803f80u;
  uint32_t xp[P][16];
  float sx[P];
  if constexpr (BITS == 4) {
#pragma unroll
    for (int c = 0; c < P; ++c) {
      float s = 0.0f;
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        const uint4 d = xd[c][t];
        xp[c][4 * t + 0] = __builtin_amdgcn_perm(d.z, d.x, 0x05040100u);
        xp[c][4 * t + 1] = __builtin_amdgcn_perm(d.z, d.x, 0x07060302u);
        xp[c][4 * t + 2] = __builtin_amdgcn_perm(d.w, d.y, 0x05040100u);
        xp[c][4 * t + 3] = __builtin_amdgcn_perm(d.w, d.y, 0x07060302u);
        s = gather_dot2(d.x, ones, s);
        s = gather_dot2(d.y, ones, s);
        s = gather_dot2(d.z, ones, s);
        s = gather_dot2(d.w, ones, s);
      }
      sx[c] = s;
    }
  }

  float acc[R];
  auto contract = [&](int c, const Pass& v) {
    if ((c * LPR + ll) * kVals >= K) { return; }
#pragma unroll
    for (int r = 0; r < R; ++r) {
      const uint32_t cw[4] = {v.c[r].x, v.c[r].y, v.c[r].z, v.c[r].w};
      const float s = bf16_bits_to_f32(v.s[r]), b = bf16_bits_to_f32(v.b[r]);
      if constexpr (BITS == 4) {
        float d = 0.0f;
#pragma unroll
        for (int t = 0; t < 4; ++t) {
#pragma unroll
          for (int i = 0; i < 4; ++i) { d = gather_dot2(xp[c][4 * t + i], ((cw[t] >> (4 * i)) & mask) | magic, d); }
        }
        acc[r] = fmaf(s, fmaf(-128.0f, sx[c], d), acc[r]);
        acc[r] = fmaf(b, sx[c], acc[r]);
      } else {
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const uint4 d = xd[c][i >> 1];
          const uint32_t x01 = (i & 1) ? d.z : d.x, x23 = (i & 1) ? d.w : d.y;
          acc[r] = fmaf(bf16_lo_to_f32(x01), fmaf(s, (float)(cw[i] & 0xffu), b), acc[r]);
          acc[r] = fmaf(bf16_hi_to_f32(x01), fmaf(s, (float)((cw[i] >> 8) & 0xffu), b), acc[r]);
          acc[r] = fmaf(bf16_lo_to_f32(x23), fmaf(s, (float)((cw[i] >> 16) & 0xffu), b), acc[r]);
          acc[r] = fmaf(bf16_hi_to_f32(x23), fmaf(s, (float)(cw[i] >> 24), b), acc[r]);
        }
      }
    }
  };
  for (;;) {
    const int next = set + stride;
    Pass nxt[kAhead];
    if constexpr (kAhead == P) {
      if (next < sets) {
#pragma unroll
        for (int c = 0; c < P; ++c) { fetch(next, c, nxt[c]); }
      }
    }
#pragma unroll
    for (int r = 0; r < R; ++r) { acc[r] = 0.0f; }
#pragma unroll
    for (int c = 0; c < P; ++c) {
      if constexpr (kAhead == P) {
        contract(c, cur[c]);
      } else {
        if (c + 1 < P || next < sets) { fetch(c + 1 < P ? set : next, c + 1 < P ? c + 1 : 0, nxt[0]); }
        contract(c, cur[0]);
        cur[0] = nxt[0];
      }
    }
    // ---- row sums ----
    if constexpr (LPR == 64) {
      const float v = row_sum(fold16(fold32(acc[0], acc[1]), fold32(acc[2], acc[3])));
      // lanes 0..15: row 0 of the set; 16..31: row 2; 32..47: row 1; 48..63: row 3
      const int r = ((lane >> 5) & 1) | ((lane >> 3) & 2), n = set * kRows + r;
      const float total = expert_ok ? v : 0.0f;
      if (gate_act) {
        const auto o = __builtin_amdgcn_permlane32_swap(__float_as_uint(total), __float_as_uint(total), false, false);
        if ((lane & 15) == 0 && lane < 32 && n + 1 < N) {            // (rows 0 and 2, with their neighbours 32 lanes up)
          y[n >> 1] = (uint16_t)f32_to_bf16_bits(gated_f32(gate_act, total, __uint_as_float(o[1])));
        }
      } else if ((lane & 15) == 0 && n < N) {
        if (ONE && y_f32) {
          static_cast<float*>(y_)[n] = total;
        } else {
          uint32_t v16 = f32_to_bf16_bits(total);
          if (ONE && residual != nullptr) { v16 = f32_to_bf16_bits(bf16_bits_to_f32(v16) + bf16_bits_to_f32(residual[n])); }
          y[n] = (uint16_t)v16;
        }
      }
    } else {
      // even rows of 16 lanes: rows 0 (a) and 2 (b) of the half's four; odd ones: 1 and 3
      const float v01 = row_sum(fold16(acc[0], acc[1])), v23 = row_sum(fold16(acc[2], acc[3]));
      const float a = expert_ok ? v01 : 0.0f, b = expert_ok ? v23 : 0.0f;
      const int odd = (lane >> 4) & 1, n = set * kRows + sub * R + odd;
      if (gate_act) {
        const float ua = __shfl_xor(a, 16, kWave), ub = __shfl_xor(b, 16, kWave);
        if ((lane & 15) == 0 && odd == 0) {
          if (n + 1 < N) { y[n >> 1] = (uint16_t)f32_to_bf16_bits(gated_f32(gate_act, a, ua)); }
          if (n + 3 < N) { y[(n + 2) >> 1] = (uint16_t)f32_to_bf16_bits(gated_f32(gate_act, b, ub)); }
        }
      } else if ((lane & 15) == 0) {
        if (n < N) { y[n] = (uint16_t)f32_to_bf16_bits(a); }
        if (n + 2 < N) { y[n + 2] = (uint16_t)f32_to_bf16_bits(b); }
      }
    }
    if (next >= sets) { break; }
    if constexpr (kAhead == P) {
#pragma unroll
      for (int c = 0; c < P; ++c) { cur[c] = nxt[c]; }
    }
    set = next;
  }
}

// One row of x against up to four packs: the workgroups of pack i start at first[i].
struct GatherRow {
  const uint16_t* x;
  const uint16_t* residual;   // (of a single pack)
  int K, gate_act, y_f32, nseg;
  QmvSeg seg[4];
  int first[5];
};

}  // namespace

template <int BITS, int P, int LPR>
__global__ __launch_bounds__(256) void qmv_gather_kernel(const uint32_t* __restrict__ w, const uint16_t* __restrict__ scales,
                                                         const uint16_t* __restrict__ biases, const uint16_t* __restrict__ x,
                                                         const int* __restrict__ pair_eid, int K, int N, int x_div, int n_experts,
                                                         uint16_t* __restrict__ y, int gate_act)
{
  gather_body<BITS, P, LPR, false>(w, scales, biases, x, pair_eid, K, N, x_div, n_experts, y, gate_act, (int)blockIdx.x,
                                   (int)gridDim.x, nullptr, 0);
}

template <int P>
__global__ __launch_bounds__(256) void qmv_gather_row8_kernel(const GatherRow p)
{
  const int at = (int)blockIdx.x;
  QmvSeg seg = p.seg[0];
  int first = 0, end = p.first[1];                          // (constant indexes: a variable one would put p into scratch)
  if (p.nseg > 1 && at >= p.first[1]) { seg = p.seg[1]; first = p.first[1]; end = p.first[2]; }
  if (p.nseg > 2 && at >= p.first[2]) { seg = p.seg[2]; first = p.first[2]; end = p.first[3]; }
  if (p.nseg > 3 && at >= p.first[3]) { seg = p.seg[3]; first = p.first[3]; end = p.first[4]; }
  gather_body<8, P, 64, true>(seg.w, seg.scales, seg.biases, p.x, nullptr, p.K, seg.N, 1, 1, seg.y, p.gate_act, at - first,
                              end - first, p.residual, p.y_f32);
}

bool qmv_gather_supports(int K, int bits) { return K % 64 == 0 && K <= (bits == 8 ? 5120 : 4096); }

namespace {

// Wavefronts of about two rounds (32 a CU), each with as many sets of its pair or pack as that leaves.  With 16 / 32 a CU, 2048 ->
// 2 x 768 at 4 tokens of 8 experts 14.6 / 13.3 us, 768 -> 2048 at 16 tokens 23.9 / 22.2.
long gather_sets_per_wave(long sets, int cus)
{
  const long room = 32L * cus;
  return (sets + room - 1) / room;
}

}  // namespace

// One row of x, up to four 8-bit packs.  Measured (us, the general kernel / now): 4096 -> 1024 5.2 / 5.1, 4096 -> 4096 7.8 / 6.8,
// 4096 -> 12288 16.6 / 14.1, 5120 -> 151936 182 / 146; gated, by qmv_rows8_kernel / now: 4096 -> 24576 29.9 / 23.9, 5120 -> 34816
// 49.3 / 38.8.
hipError_t launch_qmv_gather_row8(hipStream_t st, const QmvArgs& a, const QmvGroup& g)
{
  const int cus = a.cu_count > 0 ? a.cu_count : 256;
  GatherRow p{};
  p.x = a.x; p.residual = a.residual; p.K = a.K; p.gate_act = a.gate_act; p.y_f32 = a.y_f32 ? 1 : 0; p.nseg = g.count;
  long sets = 0;
  for (int i = 0; i < g.count; ++i) { sets += (g.seg[i].N + 3) / 4; }
  const long per = gather_sets_per_wave(sets, cus);
  for (int i = 0; i < g.count; ++i) {
    p.seg[i] = g.seg[i];
    p.first[i + 1] = p.first[i] + (int)(((g.seg[i].N + 3) / 4 + 4 * per - 1) / (4 * per));
  }
  const dim3 grid((unsigned)p.first[g.count]), block(256);
  switch ((a.K + 1023) / 1024) {
    case 1: return launch_kernel(qmv_gather_row8_kernel<1>, grid, block, 0, st, p);
    case 2: return launch_kernel(qmv_gather_row8_kernel<2>, grid, block, 0, st, p);
    case 3: return launch_kernel(qmv_gather_row8_kernel<3>, grid, block, 0, st, p);
    case 4: return launch_kernel(qmv_gather_row8_kernel<4>, grid, block, 0, st, p);
    case 5: return launch_kernel(qmv_gather_row8_kernel<5>, grid, block, 0, st, p);
    default: return hipErrorInvalidValue;
  }
}

hipError_t launch_qmv_gather(hipStream_t st, const QmvArgs& a, int bits, const int* pair_eid, int pairs, int x_div, int n_experts)
{
  const int cus = a.cu_count > 0 ? a.cu_count : 256;
  const bool half = bits == 4 && a.K <= 1024;
  const int rows = half ? 8 : 4, sets = (a.N + rows - 1) / rows;
  const long per = gather_sets_per_wave((long)sets * pairs, cus);
  const int blocks = (int)((sets + 4 * per - 1) / (4 * per));
  const dim3 grid((unsigned)blocks, (unsigned)pairs), block(256);
  uint16_t* y = reinterpret_cast<uint16_t*>(a.y);
#define VPQ_GATHER(BITS, P, LPR)                                                                                    \
  launch_kernel(qmv_gather_kernel<BITS, P, LPR>, grid, block, 0, st, a.w, a.scales, a.biases, a.x, pair_eid, a.K, a.N, \
                x_div, n_experts, y, a.gate_act)
  if (bits == 8) {
    return a.K <= 1024   ? VPQ_GATHER(8, 1, 64)
           : a.K <= 2048 ? VPQ_GATHER(8, 2, 64)
           : a.K <= 3072 ? VPQ_GATHER(8, 3, 64)
           : a.K <= 4096 ? VPQ_GATHER(8, 4, 64)
                         : VPQ_GATHER(8, 5, 64);
  }
  if (half) { return VPQ_GATHER(4, 1, 32); }
  return a.K <= 2048 ? VPQ_GATHER(4, 1, 64) : VPQ_GATHER(4, 2, 64);
#undef VPQ_GATHER
}

}  // namespace vpq
