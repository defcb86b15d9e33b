// QMM for GEMMs whose 256-row tiles would leave CUs idle (a prompt of some hundred rows, the narrow projections of a
// longer one): y[M,N] = x[M,K] . bf16(W)^T on v_mfma_f32_32x32x16, K in ascending order, fp32 accumulators, one
// rounding -- the arithmetic and the bits of the 256 x 128 tile kernel.
//
// Split.  A workgroup of four wavefronts owns 32 MT rows of x and 128 weight rows; wavefront i holds the weight rows
// [32 i, 32 (i + 1)) against all rows of x.  So every weight is unpacked once per workgroup, by the wavefront
// that multiplies it, straight into the MFMA's operand registers: no weight tile in LDS, no producer role, and the
// only thing the wavefronts share is the x tile.  Two workgroups fit a CU and fill each other's waits.  Unpacking costs
// about 2.9 vector instructions a weight, so a tile shorter than 96 rows would be bound by it.
//
// Loads.  x comes through three LDS stages of 64 values of K (direct-to-LDS, 8 rows x 128 bytes each), requested two to
// three steps ahead; one barrier a step.  Codes come 128 bytes per weight row at a time (four steps of 4 bits, two of 8),
// whole lines into a slot of the wavefront's own, which is copied to registers and requested again at once; with 8 bits into
// two slots in turn, so that a chunk is requested four steps ahead like those of 4 bits.  Scales and biases of four steps are
// one ordinary load of each per lane, requested four steps ahead.  The wait for them is the compiler's and empties the queue;
// it stands before the coming tile of x is requested.  (8 bits with one slot and that wait every second step, us, 4096 ->
// 4096 at 80 / 333 / 700 rows, packs from HBM: 38.0 / 38.3 / 41.7 -> 34.9 / 35.0 / 40.5; 12288 -> 3072 112 / 113 / 116 -> 97 / 96 /
// 105; from the shared cache 30.8 / 34.3 / 39.2 -> 30.8 / 33.4 / 39.0 and 91 / 93 / 100 -> 87 / 88 / 98.)
//
// A step is four quarters of 16 values of K.  While a quarter's MFMAs run, the wavefront reads the next quarter's fragments
// of x and unpacks its weights, one MFMA between every few vector instructions.  The barrier stands before the fourth
// quarter: by then every fragment of the step is in registers, and the first reads of the next step run under that
// quarter's MFMAs.  Read and unpacked in the quarter that uses them: 5 to 12 % slower at 80..333 rows.
//
// With K split over workgroups (few tiles over a long K) a share leaves fp32 planes that splitk_fold adds in order.
//
// What bounds it.  A workgroup alone on its CU: the LDS reads' latency, 230 cycles for a quarter of 130 (0.39 us a step at
// 64 rows; 4 bits with six stages of x and two slots of codes, without the compiler's wait: no gain).  Several to a CU: no unit
// alone -- on 4096 -> 24576 gated at 333 rows the vector ALU is busy 49 % of the cycles, the matrix pipe 40 %, LDS reads 36 %, a
// third of that bank conflicts (direct-to-LDS writes are not counted) -- but an MFMA holds the vector ALU for half of its 32
// cycles (a slot of n instructions lasts 18 + 4 n), at a clock that the power limit holds at 1.5 to 1.8 GHz.  Two 32-row
// fragments of weights a wavefront halve the LDS reads but leave half the workgroups: 2 % at 2048 tokens of experts, slower
// below 512 rows.
// Stores: lanes l and l + 32 exchange quads so that each stores 16 bytes; with four 4-byte pieces and a divide in the
// activation the store of a 128-row gated tile took 6.9 us of a workgroup's 34.
// Measured (us, fragments read where they are used, narrow stores; now): 4096 -> 24576 gated at 80 / 128 / 333 rows
// 47 / 53 / 99 -> 41 / 49 / 91; 4096 -> 4096 at 128 / 333 / 1000 rows 21.4 / 29.3 / 53.7 -> 18.2 / 26.8 / 46.4; groups of
// 32, 3840 -> 3840 at 333 rows 33.5 -> 30.0.
#include <atomic>
#include <cmath>
#include <type_traits>

#include "vpq_device.h"
#include "vpq_internal.h"
#include "vpq_tile_dequant.h"

namespace vpq {

namespace {

constexpr int kMidWaves = 4;
constexpr int kMidStages = 3;                 // stages of x
constexpr int kMidTileN = 32 * kMidWaves;     // weight rows per workgroup
constexpr int kMidRowB = 128;                 // bytes of an LDS row: 64 elements of x, or a chunk of codes

// Chunks of codes that a wavefront holds in LDS.  A chunk of 8 bits is two steps of K, too few to wait one out behind the one
// in hand; the expert-sorted form has no LDS for a second (two workgroups of five fragments fill a CU).
constexpr int mid_slots(int bits, bool grouped) { return bits == 8 && !grouped ? 2 : 1; }

struct MidParams {
  const uint32_t* w;
  const uint16_t* scales;
  const uint16_t* biases;
  const uint16_t* x;
  uint16_t* y;
  int K, N, M;
  int tiles_m, tiles_n;
  int gate_act, out_stride, out_off;          // as in the tile kernel
  int ksplit, steps_per_split;
  float* plane;                               // ksplit > 1: [ksplit][M][N]
  // Expert-sorted form: slots in blocks of kGroupedBlockRows that each belong to one expert
  // (gpu-kernels/metal/quant/affine_qmm_steel.metal:1022-1040).  tile2e[block] is the expert whose slab of the batched
  // pack [E, N, ...] the block multiplies (outside 0..n_experts - 1: nothing to do).  Gated: slot i reads x[srow[i]]
  // (outside 0..rows_x - 1: a padding slot, whose output is zero) and stores y[i].  Plain: slot i reads x[i] and
  // stores y[sdst[i]] (outside 0..rows_y - 1: not written).
  const int* tile2e;
  const int* srow;
  const int* sdst;
  int n_experts, rows_x, rows_y;
};

__device__ __forceinline__ uint32_t mid_lds(const uint8_t* q)
{
  return (uint32_t)(uintptr_t)(__attribute__((address_space(3))) const uint8_t*)q;
}

// 16 bytes per lane, global -> LDS at lds_dst + 16 * lane.  Written out by hand: the compiler orders every later LDS read
// after a direct-to-LDS load that it knows about, whatever that load fills.  The LDS base travels in M0, bound as an
// operand (the s_nop is the wait state between that write and the load, and the fifth between a base that comes back from a
// spill, v_readlane, and the load; the build checks the distance).
__device__ __forceinline__ void mid_dma16(uint32_t lds_dst, const uint8_t* base, uint32_t lane_off)
{
  const uint32_t m0v = __builtin_amdgcn_readfirstlane(lds_dst);
  asm volatile("s_nop 1\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(lane_off), "s"(base), "{m0}"(m0v) : "memory");
}

template <bool F16>
__device__ __forceinline__ floatx16 mid_mfma(u32x4 a, u32x4 b, floatx16 c)
{
  if constexpr (F16) {
    typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_32x32x16_f16(__builtin_bit_cast(halfx8, a), __builtin_bit_cast(halfx8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_32x32x16_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
}

// A workgroup's tile: rows [m0, m0 + 32 MT) of x (of slots) against weight rows [n0, n0 + 128) of the pack given, over
// share `ks` of K.
// GROUPED: `slots` holds the block's srow (gated) or sdst values, lane l of [j] that of slot 64 j + l; `span` slots are
// the workgroup's.
template <int MT, int BITS, int GROUP, bool F16, bool GROUPED>
__device__ __forceinline__ void mid_tile(const MidParams& p, uint8_t* x_lds, int m0, int n0, int ks,
                                         const uint32_t* pack_w, const uint16_t* pack_s, const uint16_t* pack_b,
                                         const int (&slots)[4], int span)
{
  constexpr int BM = 32 * MT;
  constexpr int SPC = 16 / BITS;                    // K steps of 64 per chunk of codes: 4 or 2
  constexpr int SLOTS = mid_slots(BITS, GROUPED);   // chunks of codes in LDS per wavefront
  constexpr bool kAhead = SPC * SLOTS == 4;         // a chunk is in LDS a step before its first is taken
  constexpr int SP = 4;                             // K steps per read of scales and biases
  constexpr int SG = SP * 64 / GROUP;               // groups per read
  constexpr int SGW = SG / 2;                       // ... in words of two
  constexpr int XL = MT;                            // loads of x per wavefront and step
  constexpr int CL = 4;                             // loads of codes per wavefront and chunk
  constexpr int kXStage = BM * kMidRowB;
  constexpr int kSlot = 32 * kMidRowB;
  constexpr int kWords = kMidRowB / 4 / 2;          // words of a weight row's chunk that one lane unpacks

  uint8_t* c_lds = x_lds + kMidStages * kXStage;
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int frow = lane & 31;                       // row of a 32-row operand
  const int fkh = lane >> 5;                        // which 8 of its 16 k

  const int k_first = ks * p.steps_per_split;
  const int k_left = p.K / 64 - k_first;
  const int steps = k_left < p.steps_per_split ? k_left : p.steps_per_split;
  const int chunks = (steps + SPC - 1) / SPC, reads = (steps + SP - 1) / SP;

  // ---- addresses ----
  const uint8_t* xblk = reinterpret_cast<const uint8_t*>(p.x) + (GROUPED && p.gate_act ? (size_t)0 : (size_t)m0 * p.K * 2) +
                        (size_t)k_first * 128;
  uint32_t x_off[XL];
#pragma unroll
  for (int i = 0; i < XL; ++i) {
    const int row = (wave * XL + i) * 8 + (lane >> 3);
    int rg = m0 + row < p.M ? row : p.M - 1 - m0;
    if constexpr (GROUPED) {
      if (p.gate_act) {                             // a padding slot reads row 0, unused
        const int j = (wave * XL + i) >> 3;         // (8 rows lie in one 64)
        const int at = j == 0 ? slots[0] : j == 1 ? slots[1] : j == 2 ? slots[2] : slots[3];
        const int src = __shfl(at, row & 63, kWave);
        rg = src >= 0 && src < p.rows_x ? src : 0;
      }
    }
    x_off[i] = (uint32_t)rg * (uint32_t)p.K * 2u + (uint32_t)(((lane & 7) ^ ((row >> 1) & 7)) * 16);
  }
  const int nw = n0 + wave * 32;                  // this wavefront's first weight row
  const uint32_t row_bytes = (uint32_t)p.K * BITS / 8;
  const int row_left = (int)row_bytes - k_first * (8 * BITS);   // bytes of a row from this share's start on
  const uint8_t* cblk = reinterpret_cast<const uint8_t*>(pack_w) + (size_t)(nw < p.N ? nw : p.N - 1) * row_bytes +
                        (size_t)k_first * (8 * BITS);
  const int w_last = nw < p.N ? p.N - 1 - nw : 0;   // rows past the last repeat it
  uint32_t c_lane = (uint32_t)(lane >> 3);          // load i of a chunk covers rows 8 i .. 8 i + 7
  const uint32_t c_piece = (uint32_t)(((lane & 7) ^ (lane >> 4)) * 16);   // key (row >> 1) & 7, bit 2 by the load
  const int Kg = p.K / GROUP;
  const size_t sb_at = (size_t)(nw < p.N ? nw : p.N - 1) * Kg;
  const uint16_t* sblk = pack_s + sb_at;
  const uint16_t* bblk = pack_b + sb_at;
  const uint32_t sb_row = (uint32_t)(frow < w_last ? frow : w_last) * (uint32_t)Kg;
  uint8_t* slots_c = c_lds + wave * (SLOTS * kSlot);

  auto request_x = [&](int step, int stage) {
    const uint8_t* src = xblk + (size_t)step * 128;
    const uint32_t dst = mid_lds(x_lds) + (uint32_t)(stage * kXStage + wave * (XL * 1024));
#pragma unroll
    for (int i = 0; i < XL; ++i) { mid_dma16(dst + i * 1024, src, x_off[i]); }
  };
  auto request_codes = [&](int c, int slot) {
    const uint8_t* src = cblk + (size_t)c * 128;
    const int left = row_left - c * 128;            // a piece past the row's end reads the chunk's first, unused
    const uint32_t dst = mid_lds(slots_c) + (uint32_t)(slot * kSlot);
    asm volatile("" : "+v"(c_lane));                // (no register per load is held over the loop)
#pragma unroll
    for (int i = 0; i < CL; ++i) {
      const uint32_t at = c_piece ^ (uint32_t)((i & 1) * 64);
      const uint32_t row = c_lane + 8 * i, live = row < (uint32_t)w_last ? row : (uint32_t)w_last;
      mid_dma16(dst + i * 1024, src, __umul24(live, row_bytes) + ((int)at < left ? at : 0u));
    }
  };
  uint32_t sn[SGW], bn[SGW];                        // scales and biases of the coming SP steps
  auto request_scales = [&](int c) {
    const int g0 = k_first * (64 / GROUP) + c * SG;
    if (g0 + SG <= Kg) {
      __builtin_memcpy(sn, sblk + (sb_row + (uint32_t)g0), SG * 2);
      __builtin_memcpy(bn, bblk + (sb_row + (uint32_t)g0), SG * 2);
    } else {
#pragma unroll
      for (int i = 0; i < SGW; ++i) {
        const int g = g0 + 2 * i < Kg ? g0 + 2 * i : Kg - 1, h = g0 + 2 * i + 1 < Kg ? g0 + 2 * i + 1 : Kg - 1;
        sn[i] = (uint32_t)sblk[sb_row + (uint32_t)g] | ((uint32_t)sblk[sb_row + (uint32_t)h] << 16);
        bn[i] = (uint32_t)bblk[sb_row + (uint32_t)g] | ((uint32_t)bblk[sb_row + (uint32_t)h] << 16);
      }
    }
  };

  floatx16 acc[MT];
#pragma unroll
  for (int i = 0; i < MT; ++i) {
#pragma unroll
    for (int e = 0; e < 16; ++e) { acc[i][e] = 0.0f; }
  }
  uint32_t cw[kWords], sc[SGW], bi[SGW];

  const uint32_t f_sw = (uint32_t)((frow >> 1) & 7);
  auto take_codes = [&](auto first, auto last, int slot) {   // those of the MFMAs [first, last) of a chunk
    constexpr int lo = decltype(first)::value, hi = decltype(last)::value;
    const uint8_t* rp = slots_c + slot * kSlot + frow * kMidRowB;
    if constexpr (BITS == 4) {
#pragma unroll
      for (int q = lo; q < hi; ++q) {               // MFMA q: word 2q + fkh
        cw[q] = *reinterpret_cast<const uint32_t*>(rp + (((uint32_t)(q >> 1) ^ f_sw) * 16) + (q & 1) * 8 + fkh * 4);
      }
    } else {
#pragma unroll
      for (int q = lo; q < hi; ++q) {               // MFMA q: words 4q + 2 fkh, + 1
        const u32x2 v = *reinterpret_cast<const u32x2*>(rp + (((uint32_t)q ^ f_sw) * 16) + fkh * 8);
        cw[2 * q] = v[0];
        cw[2 * q + 1] = v[1];
      }
    }
  };
  // Operands of one quarter step: the MT fragments of x and the unpacked weights, two sets in turn.
  u32x4 xf[2][MT], wf[2];
  auto read_x = [&](int stage, auto k_c) {          // quarter k of a step
    constexpr int k = decltype(k_c)::value;
    const uint8_t* xb = x_lds + stage * kXStage + frow * kMidRowB + ((uint32_t)(2 * k + fkh) ^ f_sw) * 16;
#pragma unroll
    for (int i = 0; i < MT; ++i) { xf[k & 1][i] = *reinterpret_cast<const u32x4*>(xb + i * (32 * kMidRowB)); }
  };
  auto unpack = [&](auto q_c) {                     // MFMA q of the SP steps
    constexpr int at = decltype(q_c)::value, q = at % (4 * SPC);   // q: ... of the taken chunk
    constexpr int g = at * 16 / GROUP;              // group of the taken scales
    const float s = (g & 1) ? elt_hi_to_f32<F16>(sc[g >> 1]) : elt_lo_to_f32<F16>(sc[g >> 1]);
    const float b = (g & 1) ? elt_hi_to_f32<F16>(bi[g >> 1]) : elt_lo_to_f32<F16>(bi[g >> 1]);
    uint4 wv;
    if constexpr (BITS == 4) {
      wv = dequant_word_fp8<F16>(cw[q], s, b);
    } else {
      wv = dequant_bytes(cw[2 * q], cw[2 * q + 1], s, b);
    }
    wf[q & 1] = u32x4{wv.x, wv.y, wv.z, wv.w};
  };
  auto keep = [&](auto set_c) {                     // no instruction: the unpacking stays where it is written
    u32x4& v = wf[decltype(set_c)::value];
    asm volatile("" : "+v"(v));
  };
  auto multiply = [&](auto k_c) {
    constexpr int k = decltype(k_c)::value;
#pragma unroll
    for (int i = 0; i < MT; ++i) { acc[i] = mid_mfma<F16>(wf[k & 1], xf[k & 1][i], acc[i]); }
  };
  // What a quarter interleaves: the next quarter's reads of x first, then one MFMA between the unpacking's instructions.
  auto interleave = [&]() {
    __builtin_amdgcn_sched_group_barrier(0x100, MT, 0);
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      __builtin_amdgcn_sched_group_barrier(0x008, 1, 0);
      __builtin_amdgcn_sched_group_barrier(0x002, 24 / MT, 0);
    }
  };

  // ---- K loop ----
  // Stage t % 3 holds x(t); x(t + 3) is requested once every wavefront is past step t.  A chunk of codes is requested once
  // the one before has been copied to registers.
  constexpr std::integral_constant<int, 0> kNone{};
  constexpr std::integral_constant<int, 4> kFour{};
  constexpr std::integral_constant<int, SPC * 4> kAll{};
  auto take_scales = [&]() {
#pragma unroll
    for (int i = 0; i < SGW; ++i) {
      sc[i] = sn[i];
      bi[i] = bn[i];
      asm volatile("" : "+v"(sc[i]), "+v"(bi[i]));
    }
  };
  // (the taken codes are in registers: their slot is free.)  `scales`: those from this chunk on, too.
  auto request_chunk = [&](int c, int slot, auto scales) {
    if (c < chunks) {
#pragma unroll
      for (int i = 0; i < kWords; ++i) { asm volatile("" : "+v"(cw[i])); }
      request_codes(c, slot);
      if constexpr (decltype(scales)::value) { request_scales(c / (SP / SPC)); }
    }
  };
  request_codes(0, 0);
  if (SLOTS > 1 && chunks > 1) { request_codes(1, 1); }
  request_scales(0);
  request_x(0, 0);
  for (int t = 1; t < kMidStages && t < steps; ++t) { request_x(t, t); }
  asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" : : : "memory");
  take_codes(kNone, kAll, 0);
  take_scales();
  asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
  request_chunk(SLOTS, 0, std::bool_constant<kAhead>());
  if (!kAhead && reads > 1) { request_scales(1); }
  read_x(0, kNone);
  unpack(kNone);
  keep(kNone);
  int stage = 0;
  // Step `sub` of the SP steps c: its first three quarters, then the passage to the next step, under whose cover the fourth
  // runs.
  auto step = [&](int c, auto sub_c) {
    constexpr int sub = decltype(sub_c)::value, in_chunk = sub % SPC;
    constexpr int q = sub * 4;
    constexpr int slot = sub / SPC % SLOTS, slot_next = (sub / SPC + 1) % SLOTS;
    const int t = c * SP + sub, chunk = c * (SP / SPC) + sub / SPC;
    auto quarter = [&](auto k_c) {
      constexpr int k = decltype(k_c)::value;
      __builtin_amdgcn_sched_barrier(0);
      read_x(stage, std::integral_constant<int, k + 1>());
      multiply(k_c);
      unpack(std::integral_constant<int, q + k + 1>());
      interleave();
      keep(std::integral_constant<int, (k + 1) & 1>());
      __builtin_amdgcn_sched_barrier(0);
    };
    quarter(std::integral_constant<int, 0>());
    if constexpr (kAhead && in_chunk == 0) {
      if (sub > 0 || c > 0) { request_chunk(chunk + SLOTS, slot, std::bool_constant<sub == 0>()); }
    }
    if (!kAhead && sub == 0 && c > 0 && c + 1 < reads) { request_scales(c + 1); }
    quarter(std::integral_constant<int, 1>());
    if constexpr (kAhead && in_chunk == SPC - 1) { take_codes(kNone, kFour, slot_next); }   // (there since the last passage)
    quarter(std::integral_constant<int, 2>());
    // The passage needs x(t + 1), requested two passages ago, and the next chunk's codes: a step before the chunk's end
    // (kAhead) or at it.  Younger than those are a step of x and the codes requested since the passage before last.
    if constexpr (sub == SP - 1) { take_scales(); }           // (the compiler waits for everything)
    constexpr bool kSince = SLOTS > 1 || in_chunk < SPC / 2;
    if (t + kMidStages - 1 >= steps) {
      asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" : : : "memory");
    } else if (kSince && chunk + SLOTS < chunks) {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(XL + CL) : "memory");
    } else {
      asm volatile("s_waitcnt vmcnt(%0) lgkmcnt(0)" : : "n"(XL) : "memory");
    }
    __builtin_amdgcn_s_barrier();
    asm volatile("" : : : "memory");
    if (t + kMidStages < steps) { request_x(t + kMidStages, stage); }
    stage = stage == kMidStages - 1 ? 0 : stage + 1;
    __builtin_amdgcn_sched_barrier(0);
    read_x(stage, kNone);
    if constexpr (in_chunk == SPC - 1) {
      if constexpr (kAhead) {
        take_codes(kFour, kAll, slot_next);
      } else {
        take_codes(kNone, kAll, slot_next);
      }
    }
    multiply(std::integral_constant<int, 3>());
    unpack(std::integral_constant<int, sub + 1 < SP ? q + 4 : 0>());
    if (kAhead || in_chunk < SPC - 1) { interleave(); }
    keep(kNone);
    __builtin_amdgcn_sched_barrier(0);
    // (behind the unpacking: before it, 303 us for 277 of 2048 tokens, 128 experts)
    if constexpr (!kAhead && in_chunk == SPC - 1) { request_chunk(chunk + 2, slot, std::false_type()); }
  };
  const int full = steps / SP;
  for (int c = 0; c < full; ++c) {
    step(c, std::integral_constant<int, 0>());
    step(c, std::integral_constant<int, 1>());
    step(c, std::integral_constant<int, 2>());
    step(c, std::integral_constant<int, 3>());
  }
  const int rest = steps - full * SP;
  if (rest > 0) {
    step(full, std::integral_constant<int, 0>());
    if (rest > 1) {
      step(full, std::integral_constant<int, 1>());
      if (rest > 2) { step(full, std::integral_constant<int, 2>()); }
    }
  }

  // ---- store: a lane holds, for row m = lane % 32 of each i, four consecutive n per register quad ----
  if (!GROUPED && p.ksplit > 1) {
#pragma unroll
    for (int i = 0; i < MT; ++i) {
      const int m = m0 + i * 32 + frow;
      if (m >= p.M) { continue; }
#pragma unroll
      for (int ar = 0; ar < 4; ++ar) {
        const floatx16& v = acc[i];
        const int n = nw + ar * 8 + fkh * 4;
        float* o = p.plane + ((size_t)ks * p.M + m) * p.N + n;
        if ((p.N & 3) == 0) {
          if (n < p.N) { *reinterpret_cast<floatx4*>(o) = floatx4{v[ar * 4], v[ar * 4 + 1], v[ar * 4 + 2], v[ar * 4 + 3]}; }
        } else {
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            if (n + e < p.N) { o[e] = v[ar * 4 + e]; }
          }
        }
      }
    }
    return;
  }
  // Lanes l and l + 32 hold alternate quads of one row: they exchange two of their four, and each has 16 consecutive n
  // (gated: 8 outputs) to store in 16-byte pieces.  One store also where y or its pitch is aligned to less (gfx950 takes
  // any address): 768 -> 2048 of 2048 tokens, y 8 bytes off, in 4-byte pieces 109 us against 80 of the aligned y.
  auto put = [&](uint16_t* o, u32x4 v, int left) {  // the first `left` of eight elements
    if (left >= 8) {
      __builtin_memcpy(o, &v, 16);
    } else {
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (left > 2 * e) { o[2 * e] = (uint16_t)v[e]; }
        if (left > 2 * e + 1) { o[2 * e + 1] = (uint16_t)(v[e] >> 16); }
      }
    }
  };
  auto exchange = [](uint32_t& lo, uint32_t& hi) {  // upper lanes' `lo` for lower lanes' `hi`
    const auto r = __builtin_amdgcn_permlane32_swap(lo, hi, false, false);
    lo = r[0];
    hi = r[1];
  };
#pragma unroll
  for (int i = 0; i < MT; ++i) {
    const int m = m0 + i * 32 + frow;
    bool pad = false;
    int mdst = m;
    if constexpr (GROUPED) {
      const int at = __shfl(slots[i >> 1], (i & 1) * 32 + frow, kWave);
      if (p.gate_act) {
        pad = at < 0 || at >= p.rows_x;
      } else {
        mdst = at;
        if (at < 0 || at >= p.rows_y) { continue; }
      }
    }
    if (m >= p.M) { continue; }
    const floatx16& v = acc[i];
    if (p.gate_act) {                               // (gate, up, gate, up) a quad
      uint32_t w[4];
#pragma unroll
      for (int rq = 0; rq < 4; ++rq) {
        w[rq] = pad ? 0u
                    : pack_elt2<F16>(gated_f32(p.gate_act, v[rq * 4], v[rq * 4 + 1]),
                                     gated_f32(p.gate_act, v[rq * 4 + 2], v[rq * 4 + 3]));
      }
      exchange(w[0], w[2]);
      exchange(w[1], w[3]);
      const int col = nw / 2 + fkh * 8;
      put(p.y + (size_t)m * p.out_stride + p.out_off + col, u32x4{w[0], w[2], w[1], w[3]}, p.N / 2 - col);
    } else {
      uint32_t w[8];
#pragma unroll
      for (int e = 0; e < 8; ++e) { w[e] = pack_elt2<F16>(v[2 * e], v[2 * e + 1]); }
      exchange(w[0], w[4]);
      exchange(w[1], w[5]);
      exchange(w[2], w[6]);
      exchange(w[3], w[7]);
      const int n = nw + fkh * 16;
      uint16_t* o = p.y + (size_t)mdst * p.N + n;
      put(o, u32x4{w[0], w[1], w[4], w[5]}, p.N - n);
      put(o + 8, u32x4{w[2], w[3], w[6], w[7]}, p.N - n - 8);
    }
  }
  if constexpr (GROUPED) {                          // slots past the fragments that were multiplied: padding, act(0) * 0 = +0
    if (p.gate_act) {
      for (int row = BM + frow; row < span; row += 32) {
        const int col = nw / 2 + fkh * 8;
        put(p.y + (size_t)(m0 + row) * p.out_stride + p.out_off + col, u32x4{0u, 0u, 0u, 0u}, p.N / 2 - col);
      }
    }
  }
}

}  // namespace

constexpr size_t mid_lds_bytes(int mt, int slots) { return (size_t)(kMidStages * 32 * mt + slots * kMidWaves * 32) * kMidRowB; }

template <int MT, int BITS, int GROUP, bool F16>
__global__ __launch_bounds__(kMidWaves * 64, 2) void qmm_mid_kernel(const MidParams p)
{
  constexpr int BM = 32 * MT, BN = kMidTileN;
  extern __shared__ __attribute__((aligned(16))) uint8_t x_lds[];

  // Workgroups go to the XCDs round robin: those that share a weight tile (one per tile of rows of x) are eight apart,
  // so that the pack is read from HBM once.
  const int units = p.tiles_n * p.ksplit;
  const int span = 8 * p.tiles_m;
  const int uq = (int)blockIdx.x / span, ur = (int)blockIdx.x - uq * span;
  const int unit = uq * 8 + (ur & 7);
  if (unit >= units) { return; }
  const int ks = unit / p.tiles_n;
  const int m0 = (ur >> 3) * BM, n0 = (unit - ks * p.tiles_n) * BN;
  // (the last tile multiplies as many fragments as have rows)
  const int none[4] = {}, frags = (p.M - m0 + 31) / 32;
  if (MT > 3 && frags == 3) {
    mid_tile<3, BITS, GROUP, F16, false>(p, x_lds, m0, n0, ks, p.w, p.scales, p.biases, none, 0);
  } else if (MT > 2 && frags == 2) {
    mid_tile<2, BITS, GROUP, F16, false>(p, x_lds, m0, n0, ks, p.w, p.scales, p.biases, none, 0);
  } else if (frags == 1) {
    mid_tile<1, BITS, GROUP, F16, false>(p, x_lds, m0, n0, ks, p.w, p.scales, p.biases, none, 0);
  } else {
    mid_tile<MT, BITS, GROUP, F16, false>(p, x_lds, m0, n0, ks, p.w, p.scales, p.biases, none, 0);
  }
}

// The expert-sorted form.  An expert's last block is mostly padding (16384 pairs of 128 experts: 191 blocks, 63 of them
// with about ten live slots), and a prompt of some tokens gives each expert a few: a block multiplies as many 32-row
// fragments as reach its last live slot, each count a K loop of its own, whose loads, LDS reads and MFMAs are those
// rows' alone.  A last block of one fragment is multiplied by the block before it as a fifth, so its weights are neither
// read nor unpacked a second time (two fragments would leave one workgroup per CU).  All weight tiles of a block go to one
// XCD (eight workgroups apart), whose L2 then holds its rows of x.
// Two neighbouring blocks to an XCD, which mostly share an expert's weight tiles: 1 to 2 % slower (2048 tokens 298 -> 305 us).
// WIDE or not is chosen on the host (qmm_grouped_wide).  Not WIDE is for a few tokens, where almost every block has one or
// two fragments: no loop over more of them, hence registers and LDS for three workgroups per CU instead of two, and the blocks
// that have more are multiplied half after half.  (A fourth workgroup needs spills and gains 2 % at most.)
// Bound by the plain tile's step at full blocks, by unpacking and the codes' read at one fragment.  Measured (us, sort +
// gate|up + down of one layer, 2048 -> 768; every block by itself, the plain tile's first form, four launches of the sort;
// now): 8 of 128 experts, 2048 / 512 / 64 tokens 309 / 163 / 147 -> 262 / 135 / 117; 8 bits, 2048 tokens 357 -> 319, and gate|up
// + down with the scales read every four steps instead of two, 64 / 512 / 2048 tokens 139 / 154 / 310 -> 130 / 140 / 300.
template <int BITS, bool WIDE>
__global__ __launch_bounds__(kMidWaves * 64, WIDE ? 2 : 3) void qmm_mid_grouped_kernel(const MidParams p)
{
  extern __shared__ __attribute__((aligned(16))) uint8_t x_lds[];
  static_assert(kGroupedBlockRows == 128, "two slots per lane, four fragments");

  const int span = 8 * p.tiles_n;
  const int uq = (int)blockIdx.x / span, ur = (int)blockIdx.x - uq * span;
  const int tm = uq * 8 + (ur & 7);
  if (tm >= p.tiles_m) { return; }
  const int m0 = tm * kGroupedBlockRows, n0 = (ur >> 3) * kMidTileN;
  const int lane = threadIdx.x & 63;
  const int* idx = p.gate_act ? p.srow : p.sdst;
  const int lim = p.gate_act ? p.rows_x : p.rows_y;
  const bool next = tm + 1 < p.tiles_m;
  const int slots[4] = {idx[m0 + lane], idx[m0 + 64 + lane], next ? idx[m0 + 128 + lane] : -1,
                        next ? idx[m0 + 192 + lane] : -1};
  const int e = p.tile2e[tm], e_before = tm > 0 ? p.tile2e[tm - 1] : -1;
  const int e_next = next ? p.tile2e[tm + 1] : -1, e_after = tm + 2 < p.tiles_m ? p.tile2e[tm + 2] : -1;
  if (e < 0 || e >= p.n_experts) { return; }        // the whole workgroup, before any barrier
  auto fragments = [&](int v0, int v1) {            // of a block, up to its last live slot
    const unsigned long long lo = __ballot(v0 >= 0 && v0 < lim), hi = __ballot(v1 >= 0 && v1 < lim);
    return hi != 0 ? ((hi >> 32) != 0 ? 4 : 3) : (lo >> 32) != 0 ? 2 : 1;
  };
  const int live = fragments(slots[0], slots[1]);
  if (WIDE && e_before == e && e_next != e && live == 1) { return; }   // the block before multiplies it
  const bool both = e_next == e && e_after != e && fragments(slots[2], slots[3]) == 1;

  const uint32_t* w = p.w + (size_t)e * (size_t)p.N * (size_t)(p.K >> (BITS == 4 ? 3 : 2));
  const uint16_t* s = p.scales + (size_t)e * (size_t)p.N * (size_t)(p.K >> 6);
  const uint16_t* b = p.biases + (size_t)e * (size_t)p.N * (size_t)(p.K >> 6);
  if constexpr (!WIDE) {
    int half[4] = {slots[0], -1, -1, -1};
    if (live == 1) {
      mid_tile<1, BITS, 64, false, true>(p, x_lds, m0, n0, 0, w, s, b, half, kGroupedBlockRows);
      return;
    }
    for (int h = 0; h < 2; ++h) {
      mid_tile<2, BITS, 64, false, true>(p, x_lds, m0 + h * 64, n0, 0, w, s, b, half, live == 2 ? kGroupedBlockRows : 64);
      if (live == 2) { return; }
      half[0] = slots[1];
      __builtin_amdgcn_s_barrier();                 // (nobody reads the first half's x any more)
      asm volatile("" : : : "memory");
    }
    return;
  }
  if (both) {
    mid_tile<5, BITS, 64, false, true>(p, x_lds, m0, n0, 0, w, s, b, slots, 2 * kGroupedBlockRows);
  } else if (live == 1) {
    mid_tile<1, BITS, 64, false, true>(p, x_lds, m0, n0, 0, w, s, b, slots, kGroupedBlockRows);
  } else if (live == 2) {
    mid_tile<2, BITS, 64, false, true>(p, x_lds, m0, n0, 0, w, s, b, slots, kGroupedBlockRows);
  } else if (live == 3) {
    mid_tile<3, BITS, 64, false, true>(p, x_lds, m0, n0, 0, w, s, b, slots, kGroupedBlockRows);
  } else {
    mid_tile<4, BITS, 64, false, true>(p, x_lds, m0, n0, 0, w, s, b, slots, kGroupedBlockRows);
  }
}

// y[i] = elt(plane[0][i] + plane[1][i] + ...) in that order, four at a time where the count allows.
template <int VEC>
__global__ __launch_bounds__(256) void splitk_fold_kernel(const float* __restrict__ plane, uint16_t* __restrict__ y,
                                                          size_t count, int splits)
{
  for (size_t i = ((size_t)blockIdx.x * 256 + threadIdx.x) * VEC; i < count; i += (size_t)gridDim.x * 256 * VEC) {
    if constexpr (VEC == 4) {
      floatx4 v = *reinterpret_cast<const floatx4*>(plane + i);
      for (int s = 1; s < splits; ++s) { v += *reinterpret_cast<const floatx4*>(plane + (size_t)s * count + i); }
      *reinterpret_cast<uint2*>(y + i) = make_uint2(pack_bf16x2(v[0], v[1]), pack_bf16x2(v[2], v[3]));
    } else {
      float v = plane[i];
      for (int s = 1; s < splits; ++s) { v += plane[(size_t)s * count + i]; }
      y[i] = (uint16_t)f32_to_bf16_bits(v);
    }
  }
}

namespace {

// More LDS than the default limit needs the attribute, set once per kernel (two threads may both set it, which is harmless).
template <typename Kernel>
hipError_t mid_launch_one(Kernel kern, std::atomic<bool>& ready, size_t lds, dim3 grid, hipStream_t st, const MidParams& p)
{
  if (!ready.load(std::memory_order_acquire)) {
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, (int)lds);
    if (e != hipSuccess) { return e; }
    ready.store(true, std::memory_order_release);
  }
  return launch_kernel(kern, grid, dim3(kMidWaves * 64), lds, st, p);
}

template <int BITS, bool WIDE>
hipError_t mid_launch_grouped(dim3 grid, hipStream_t st, const MidParams& p)
{
  static std::atomic<bool> ready{false};
  return mid_launch_one(qmm_mid_grouped_kernel<BITS, WIDE>, ready,
                        mid_lds_bytes(WIDE ? kGroupedBlockRows / 32 + 1 : 2, mid_slots(BITS, true)), grid, st, p);
}

template <int MT, int BITS, int GROUP, bool F16>
hipError_t mid_launch_rows(hipStream_t st, const MidParams& p, dim3 grid)
{
  static std::atomic<bool> ready{false};
  return mid_launch_one(qmm_mid_kernel<MT, BITS, GROUP, F16>, ready, mid_lds_bytes(MT, mid_slots(BITS, false)), grid, st, p);
}

template <int BITS, int GROUP, bool F16>
hipError_t mid_launch(hipStream_t st, const MidParams& p, int mt, dim3 grid)
{
  if (mt == 2) { return mid_launch_rows<2, BITS, GROUP, F16>(st, p, grid); }
  if (mt == 3) { return mid_launch_rows<3, BITS, GROUP, F16>(st, p, grid); }
  return mid_launch_rows<4, BITS, GROUP, F16>(st, p, grid);
}

hipError_t mid_launch_as(hipStream_t st, const GemmArgs& a, int mt, int splits, float* plane)
{
  if (a.lora_t != nullptr) { return hipErrorInvalidValue; }
  MidParams p{};
  p.w = a.w; p.scales = a.scales; p.biases = a.biases; p.x = a.x; p.y = a.y;
  p.K = a.K; p.N = a.N; p.M = a.M;
  p.gate_act = a.gate_act;
  p.out_stride = a.out_stride > 0 ? a.out_stride : a.N / 2;
  p.out_off = a.out_off;
  p.tiles_m = (a.M + 32 * mt - 1) / (32 * mt);
  p.tiles_n = (a.N + kMidTileN - 1) / kMidTileN;
  const int steps = a.K / 64;
  p.steps_per_split = (steps + splits - 1) / splits;
  p.ksplit = (steps + p.steps_per_split - 1) / p.steps_per_split;
  p.plane = plane;
  const dim3 grid((unsigned)(((long)p.tiles_n * p.ksplit + 7) / 8 * 8 * p.tiles_m));
  if (a.bits == 8) { return a.group == 64 && !a.f16 ? mid_launch<8, 64, false>(st, p, mt, grid) : hipErrorInvalidValue; }
  if (a.group == 32) { return a.f16 ? hipErrorInvalidValue : mid_launch<4, 32, false>(st, p, mt, grid); }
  return a.f16 ? mid_launch<4, 64, true>(st, p, mt, grid) : mid_launch<4, 64, false>(st, p, mt, grid);
}

// What a GEMM takes, in microseconds.  Fitted to 98 000 timings of every kernel here on 11 700 shapes, drawn ones and those of
// models (512..17408 x 512..34816 at 65..4096 rows, all four formats, plain and gated stores, 4-bit shares of K), each with a
// pack that the shared cache holds and with one that it does not: first to the times, then, under the choices that the tests
// pin, to the time of what is chosen, which is what the figures are for (the times themselves are met to 5..9 %).  On 3500 other
// drawn shapes the choice takes 0.2 % longer than the fastest kernel (mean; 2 % of the shapes 3 % and more, the worst 15 %), with
// gated stores 0.4 %, with K split 0.7 %.
//
// A split writes its planes once more, reads them once more, and folds them in a launch of its own.
double planes_us(int N, int M, int splits)
{
  return splits > 1 ? 1.9 + 0.27 * splits + (splits + 0.5) * (double)M * (double)N * 4.0 / 4.83e6 : 0.0;
}

constexpr int kXcds = 8;

enum CostFormat { kCost4, kCost8, kCostG32, kCostF16 };

// Shape of a call, as far as its time goes.
struct CostShape { int K, N, M; CostFormat format; bool gated; };

// This kernel, by the n workgroups (not a whole number) that a CU of the busiest XCD gets, since all workgroups of a weight
// tile are on one.  64 of K take lone + lone_n n while each has a CU to itself, base + more n + whole ceil(n) from then on
// (the clock falls as the load rises, and a workgroup that is left over runs alone); every ceil(n) costs a `store` (or
// `gated` store).  Every weight tile reads all of x, at 8 TB/s from the shared cache, less as more weight tiles of an XCD are in
// flight together and find each other's rows in its L2; that bounds M in the thousands.
struct MidCost { double fixed, lone, lone_n, base, more, whole, store, gated; };
constexpr MidCost kMidCost[5] = {{}, {}, {5.18, 0.3444, 0.0821, 0.1451, 0.0996, 0.1872, 0.472, 0.678},
                                 {5.64, 0.4710, 0.0338, 0.0697, 0.1331, 0.2497, 0.649, 1.364},
                                 {5.75, 0.4590, 0.0810, 0.0486, 0.2092, 0.2615, 1.342, 2.324}};
// By format.  8 bits were fitted again when their step changed: on 1560 drawn shapes with packs from HBM the choice takes 0.47 %
// longer than the fastest kernel (0.56 by the figures before); 15 shapes changed kernel, to 0.91 of their time.
constexpr double kMidLone[4] = {1.0, 1.08, 0.970, 0.886}, kMidBusy[4] = {1.0, 1.185, 0.986, 1.023};

double mid_us(const CostShape& s, int mt, int splits, int cus)
{
  const MidCost& c = kMidCost[mt];
  const int steps = s.K / 64, per = (steps + splits - 1) / splits;
  const int per_xcd = cus >= kXcds ? cus / kXcds : 1;
  const long tiles_n = (s.N + kMidTileN - 1) / kMidTileN, tiles_m = (s.M + 32 * mt - 1) / (32 * mt);
  const long wgs = (tiles_n * splits + kXcds - 1) / kXcds * tiles_m;
  const long whole = (wgs + per_xcd - 1) / per_xcd;
  const double n = (double)wgs / per_xcd;
  double step = (c.lone + c.lone_n * (n < 1.0 ? n : 1.0)) * kMidLone[s.format];
  if (n > 1.0) {
    const double busy = (c.base + c.more * n + c.whole * (double)whole) * kMidBusy[s.format];
    if (busy > step) { step = busy; }
  }
  const double us = per * step + (double)whole * (s.gated ? c.gated : c.store);
  double together = 2.0 * per_xcd / tiles_m;        // weight tiles of an XCD that are in flight (two workgroups a CU)
  const double most = (double)((tiles_n + kXcds - 1) / kXcds);
  together = together > most ? most : together < 1.0 ? 1.0 : together;
  const double fetch = (double)tiles_n * (double)s.M * (double)s.K * 2.0 / 7.97e6 / sqrt(sqrt(together));
  return c.fixed + sqrt(sqrt(us * us * us * us + fetch * fetch * fetch * fetch)) + planes_us(s.N, s.M, splits);
}

// Rows of x per workgroup, in 32s: the count that takes least.
int mid_rows(const CostShape& s, int splits, int cus)
{
  int best = 4;
  for (int mt = 3; mt >= 2; --mt) {
    if (mid_us(s, mt, splits, cus) < mid_us(s, best, splits, cus)) { best = mt; }
  }
  return best;
}

// The kernels with 256 rows of x a workgroup, one workgroup per CU: 64 of K and the store of a full chip's tiles, a round
// that leaves CUs idle takes `part` of them and up (the clock rises as the load falls).
struct TallCost { int width; double fixed, step, store, gated, part, by_format[4]; };
constexpr TallCost kTileCost = {128, 3.95, 1.085, 4.93, 7.98, 0.7586, {1.0, 1.14, 0.991, 1.070}};
constexpr TallCost kBigCost[3] = {{256, 5.72, 1.492, 5.93, 23.45, 0.8034, {1.0, 0.0, 0.994, 1.046}},     // (0: not built)
                                  {192, 4.97, 1.283, 5.53, 14.48, 0.7515, {1.0, 1.143, 0.0, 1.044}},
                                  {128, 4.26, 1.035, 3.57, 8.10, 0.8120, {1.0, 1.04, 1.003, 1.085}}};

// tiles: what the busiest CU's share comes to on the whole chip.
double tall_us(const TallCost& c, const CostShape& s, int splits, int cus, long tiles)
{
  const int steps = s.K / 64, per = (steps + splits - 1) / splits;
  const long full = tiles / cus;
  const double rest = (double)(tiles - full * cus) / cus;
  const double rounds = (double)full + (rest > 0.0 ? c.part + (1.0 - c.part) * rest * rest : 0.0);
  return c.fixed + (per * c.step * c.by_format[s.format] + (s.gated ? c.gated : c.store)) * rounds + planes_us(s.N, s.M, splits);
}

double tile_us(const CostShape& s, int splits, int cus)
{
  const long tiles = (long)((s.M + 255) / 256) * ((s.N + kTileCost.width - 1) / kTileCost.width);
  return tall_us(kTileCost, s, splits, cus, tiles * splits);
}

bool tile_splits_better(const CostShape& s, int splits, int cus)
{
  return tile_us(s, splits, cus) < mid_us(s, mid_rows(s, splits, cus), splits, cus);
}

CostShape cost_shape(const GemmArgs& a)
{
  const CostFormat f = a.bits == 8 ? kCost8 : a.group == 32 ? kCostG32 : a.f16 ? kCostF16 : kCost4;
  return CostShape{a.K, a.N, a.M, f, a.gate_act != 0};
}

// The kernel that takes least without a split of K (for the large tile: its width too), and how long.
GemmChoice choose_unsplit(const GemmArgs& a, double* us)
{
  const int cus = a.cu_count > 0 ? a.cu_count : 256;
  const CostShape s = cost_shape(a);
  const int tm = (a.M + 255) / 256;
  GemmChoice best{GemmKernel::kTile, 0};
  *us = tile_us(s, 1, cus);
  if (a.lora_t != nullptr) {                        // with an adapter: the large tile from one round of its tiles on
    const int bn = qmm_big_tile_n(a.N, a.M, cus);
    if (qmm_big_supports(a) && (long)tm * ((a.N + bn - 1) / bn) >= cus) { best = {GemmKernel::kBig, bn}; }
    return best;
  }
  const double mid = mid_us(s, mid_rows(s, 1, cus), 1, cus);
  if (mid <= *us) { best.kernel = GemmKernel::kMid; *us = mid; }
  if (!qmm_big_supports(a)) { return best; }
  for (const TallCost& c : kBigCost) {
    if (c.by_format[s.format] == 0.0) { continue; }
    const double big = tall_us(c, s, 1, cus, qmm_big_tiles_load(tm, (a.N + c.width - 1) / c.width));
    if (big < *us) { best = {GemmKernel::kBig, c.width}; *us = big; }
  }
  return best;
}

}  // namespace

GemmChoice qmm_choose(const GemmArgs& a)
{
  double us;
  return choose_unsplit(a, &us);
}

int qmm_plan(const GemmArgs& a, int splits)
{
  const int cus = a.cu_count > 0 ? a.cu_count : 256;
  const CostShape s = cost_shape(a);
  if (splits > 1) { return tile_splits_better(s, splits, cus) ? 256 : 32 * mid_rows(s, splits, cus); }
  const GemmChoice c = qmm_choose(a);
  return c.kernel == GemmKernel::kBig ? -c.width : c.kernel == GemmKernel::kTile ? 256 : 32 * mid_rows(s, 1, cus);
}

hipError_t launch_qmm_mid(hipStream_t st, const GemmArgs& a)
{
  const int cus = a.cu_count > 0 ? a.cu_count : 256;
  return mid_launch_as(st, a, mid_rows(cost_shape(a), 1, cus), 1, nullptr);
}

// Three narrow workgroups per CU instead of two wide ones where the experts' first blocks alone are more than the wide ones'
// first round, and up to 32 pairs per expert on average.  Wide against narrow, us of gate|up and down, 2048 -> 768, 8 of 128
// experts: 64 tokens (4 pairs an expert) 88 + 38 against 82 + 33, 512 (32) 93 + 44 against 86 + 38, 768 (48) 100 + 51 against 106 +
// 50, 1024 112 + 55 against 138 + 66; within one round, 2048 -> 512, 64 experts, 512 tokens, gate|up 29.3 against 30.3.
// A down projection knows its pairs (rows_y).  A gated one has its tokens and the map: as the sort leaves it, a block an expert and
// the whole blocks of all pairs; cut down to the blocks in use it says little, and the pairs are taken to be 8 a token.
bool qmm_grouped_wide(const GemmArgs& a, const GroupedArgs& g)
{
  const long cus = a.cu_count > 0 ? a.cu_count : 256, E = g.n_experts;
  if (E * ((a.N + kMidTileN - 1) / kMidTileN) <= 2 * cus) { return true; }
  if (!a.gate_act) { return (long)g.rows_y > 32 * E; }
  const long blocks = a.M / kGroupedBlockRows, tokens = g.rows_x;
  const bool whole_map = blocks - E >= (tokens + kGroupedBlockRows - 1) / kGroupedBlockRows;   // (at least a pair a token)
  return whole_map ? (blocks - E) * kGroupedBlockRows > 32 * E : tokens * 8 > 32 * E;
}

hipError_t launch_qmm_grouped(hipStream_t st, const GemmArgs& a, const GroupedArgs& g)
{
  // gated blocks gather rows of x, plain ones scatter rows of y
  if ((a.gate_act ? g.srow : g.sdst) == nullptr || (!a.gate_act && g.srow != nullptr)) { return hipErrorInvalidValue; }
  MidParams p{};
  p.w = a.w; p.scales = a.scales; p.biases = a.biases; p.x = a.x; p.y = a.y;
  p.K = a.K; p.N = a.N; p.M = a.M;
  p.gate_act = a.gate_act;
  p.out_stride = a.out_stride > 0 ? a.out_stride : a.N / 2;
  p.out_off = a.out_off;
  p.tiles_m = a.M / kGroupedBlockRows;              // a.M is a whole number of blocks
  p.tiles_n = (a.N + kMidTileN - 1) / kMidTileN;
  p.ksplit = 1; p.steps_per_split = a.K / 64;
  p.tile2e = g.tile2e; p.srow = g.srow; p.sdst = g.sdst;
  p.n_experts = g.n_experts; p.rows_x = g.rows_x; p.rows_y = g.rows_y;
  const dim3 grid((unsigned)((p.tiles_m + 7) / 8 * 8 * p.tiles_n));
  const bool wide = qmm_grouped_wide(a, g);
  if (wide) { return a.bits == 8 ? mid_launch_grouped<8, true>(grid, st, p) : mid_launch_grouped<4, true>(grid, st, p); }
  return a.bits == 8 ? mid_launch_grouped<8, false>(grid, st, p) : mid_launch_grouped<4, false>(grid, st, p);
}

// Shares of K that pay for their planes; 1 where the tiles alone fill the chip.
int qmm_choose_splits(int K, int N, int M, int cu_count)
{
  const int cus = cu_count > 0 ? cu_count : 256;
  const int steps = K / 64;
  GemmArgs a{};
  a.K = K; a.N = N; a.M = M; a.cu_count = cus;
  const CostShape shape = cost_shape(a);
  double best_us;
  choose_unsplit(a, &best_us);
  int best = 1;
  best_us *= 0.95;
  for (int s = 2; s <= 16 && steps / s >= 4; ++s) {
    const int per = (steps + s - 1) / s;
    if ((steps + per - 1) / per != s) { continue; }    // shares would come out uneven: another count covers it
    const double us = tile_splits_better(shape, s, cus) ? tile_us(shape, s, cus)
                                                        : mid_us(shape, mid_rows(shape, s, cus), s, cus);
    if (us < best_us) { best = s; best_us = us; }
  }
  return best;
}

// The count that an automatic split may not go without room for: two and more where 256 x 128 tiles that fill less than
// half of the chip would take a tenth longer unsplit (0.9 us a step of 64, 3 us a round, planes at 4 TB/s).  Callers without a
// workspace are refused there and nowhere else.
int qmm_required_splits(int K, int N, int M, int cu_count)
{
  const int cus = cu_count > 0 ? cu_count : 256;
  const int steps = K / 64, tiles = ((M + 255) / 256) * ((N + 127) / 128);
  if (tiles * 2 > cus) { return 1; }
  int best = 1;
  double best_us = 3.0 + 0.9 * steps;
  for (int s = 2; s <= 16 && steps / s >= 4; ++s) {
    const int per = (steps + s - 1) / s;
    if ((steps + per - 1) / per != s) { continue; }
    const double us = (tiles * s + cus - 1) / cus * (3.0 + 0.9 * per) + 3.0 + (s + 0.5) * (double)M * (double)N * 1e-6;
    if (us < 0.9 * best_us) { best = s; best_us = us; }
  }
  return best;
}

size_t qmm_splitk_workspace_bytes(int K, int N, int M, int cu_count)
{
  const int s = qmm_choose_splits(K, N, M, cu_count);
  return s > 1 ? (size_t)s * (size_t)M * (size_t)N * sizeof(float) : 0;
}

hipError_t launch_qmm_splitk(hipStream_t st, const GemmArgs& a, int splits, float* plane)
{
  const int cus = a.cu_count > 0 ? a.cu_count : 256;
  const int steps = a.K / 64, per = (steps + splits - 1) / splits;
  const hipError_t e = tile_splits_better(cost_shape(a), splits, cus)
                           ? launch_qmm_tile_planes(st, a, splits, plane)
                           : mid_launch_as(st, a, mid_rows(cost_shape(a), splits, cus), splits, plane);
  if (e != hipSuccess) { return e; }
  const size_t count = (size_t)a.M * (size_t)a.N;
  const bool quads = (count & 3) == 0;
  size_t blocks = (count + (quads ? 1023 : 255)) / (quads ? 1024 : 256);
  if (blocks > 65536) { blocks = 65536; }
  const int shares = (steps + per - 1) / per;
  return quads ? launch_kernel(splitk_fold_kernel<4>, dim3((unsigned)blocks), dim3(256), 0, st, plane, a.y, count, shares)
               : launch_kernel(splitk_fold_kernel<1>, dim3((unsigned)blocks), dim3(256), 0, st, plane, a.y, count, shares);
}

}  // namespace vpq
