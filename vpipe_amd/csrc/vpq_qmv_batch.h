// QMV for a batch of rows (2..64 rows of x; one row where the one-row kernel does not run), any K that is a multiple
// of 64 (of 32 for groups of 32): the kernel template of vpq_qmv_batch*.hip.
//
// What bounds it.  Up to 8 rows the pack's read and the start of a launch (4096 -> 24576 at 4 rows 14.6 us, 57 MB).  Above,
// the instructions and a workgroup's own start and end: of 36 000 cycles of three tiles and 48 rows over K = 4096, 7 800 pass
// before the first codes are there, 2 500 a piece of 64 values (two wavefronts a SIMD; 1 470 if they only issued: unpacking
// costs 18 instructions per 16 x 64 codes, every 16 x 16 outputs 8 multiply-adds per group, an MFMA holds the vector ALU for
// 8 of its 16 cycles), the rest are the end's.  x comes in once per workgroup, so it also counts how many weight rows share
// it and how many workgroups a CU gets one after the other: batch_plan. Tried: workgroups that walk over the blocks of weight
// rows and request the next block's codes and scales early (30.5 -> 28.7 us at 48 rows, but level on the mean of 7000 shapes,
// and scalar registers spill); the next piece of x read from LDS while one is contracted (28.7 -> 30.6); several pieces of x
// in flight (LDS reads take 450 cycles instead of 200 while they come in: 8 % slower); three tiles in 128 registers, two
// workgroups to a CU (4 rows 14.6 -> 17.1); x in registers (15.4 -> 18.7 at 4 rows; 104 -> 99 on 5120 -> 151936 at 8); more
// chunks in flight for 4 bits (the first arrives later: 4096 -> 4096 5.0 -> 5.5). Measured (us, before / now; before: up to
// 32 rows and two tiles a workgroup): 4096 -> 4096 at 16 / 24 / 48 rows 6.3 / 7.6 / 9.6 -> 6.0 / 7.1 / 9.6; 4096 -> 1024 at
// 24 / 48 rows 7.3 / 7.5 -> 5.4 / 6.0; 12288 -> 4096 at 16 / 24 rows 13.4 / 17.9 -> 12.1 / 15.6; 4096 -> 24576 at 4 / 48 rows
// 15.2 / 38.7 -> 14.7 / 30.5; 17408 -> 5120 at 48 / 64 rows 51 / 53 -> 34 / 35.
//
// Split.  A workgroup of eight wavefronts owns T tiles of 16 weight rows and up to 64 rows of x.  K is cut into chunks
// of 128 bytes of codes per row (256 values of 4 bits, 128 of 8 bits); chunk c belongs to wavefront c % 8, which
// contracts it for all T tiles and all rows of x.  The eight partial results meet in LDS once, at the end, in
// wavefront order.  So a result depends on K and the format alone -- not on M, N, T or the launch it is part of: a row
// of x has the same bits in a batch of any size, and a grouped launch the bits of separate ones.
//
// Loads.  Codes and x arrive by 128-bit direct-to-LDS loads into one slot per wavefront, laid out so that eight consecutive
// lanes cover one 128-byte line (an L1 has about 72 requests in flight, so what counts is bytes per request).  A slot is
// copied to registers (codes, x as MFMA operands, scales, biases), re-requested for the wavefront's next chunk, and only then
// the copy is contracted: one chunk per wavefront is always in flight and no wait has to be counted.  A workgroup with a CU
// to itself may take pieces of x twice as long (a wait, a read and a start of the contraction fewer: 12288 -> 4096 at 16 rows
// 13.1 -> 12.1 us) or, with 8 bits and a long K (twelve chunks a wavefront at 12288), two or three slots (12288 -> 4096 at 6
// rows 15.8 -> 14.4).  The 16-byte pieces of a row are XOR-swizzled so that the operand reads do not collide on banks.  The
// scales and biases of the workgroup's rows are two contiguous blocks of the pack and are brought in whole, before anything
// else.
//
// Math.  Codes become q itself in the element type (exact).  4 bits: against an accumulator seeded with -8 sum(x) of the
// group, then y += scale * sum(x (q - 8)) + (bias + 8 scale) * sum(x) in fp32; 8 bits: y += scale * sum(x q) +
// bias * sum(x) -- the factored form of gpu-kernels/metal/quant/affine_qmv.metal:151-174.  The weight is never rounded.
// The error is that of the plain sum of x * fma(scale, q, bias) (2-norm against float64, N(0,1) x, K = 3840 / 9664:
// 4 bits 0.84 / 1.02e-7 against 0.82 / 1.05, groups of 32 0.87 / 1.06 against 0.81 / 1.04, binary16 0.9 / 1.0 against
// 1.5 / 2.2, 8 bits 1.2 / 1.4 against 1.3 / 2.0).  With codes as 128 + q by one v_and_or_b32 per pair, as many
// instructions and 2 to 4 % less time, it was five times that: the sum cancels against 128 sum(x).
// An output that this form leaves non-finite (an infinity in x meets the seed's opposite infinity, or a code of zero;
// finite x near the end of the range) is summed again as x * fma(scale, q, bias) in fp32: +-inf where the plain sum gives +-inf.
//
// No inline-assembly VALU instruction may sit near the MFMAs (the compiler's hazard recogniser cannot see what such a
// statement writes); the asm here is waits only.
#pragma once

#include <atomic>
#include <cstddef>
#include <type_traits>

#include "vpq_device.h"
#include "vpq_internal.h"

namespace vpq {

constexpr int kBatchWaves = 8;

struct BatchParams {
  const uint32_t* w;
  const uint16_t* scales;
  const uint16_t* biases;
  const uint16_t* x;
  int K, N, M;
  int blocks;           // workgroups along N, all packs together
  int m_tiles;          // workgroups along M
  int rows;             // rows of x per workgroup
  // ---- not preloaded ----
  void* y;
  const uint16_t* residual;
  int gate_act;         // rows are interleaved gate|up; y is [M, N/2] = act(gate) * up (1 SwiGLU, 2 GEGLU)
  int y_f32;
  int nseg;             // packs that share x; the first is (w, scales, biases, N, y)
  QmvSeg seg[3];        // the others
  int seg_first[3];     // their first workgroup
};
// What a launch runs: tiles of 16 weight rows and rows of x (4 mr at most) of a workgroup, workgroups along M, depth.
struct BatchPlan {
  int tiles, mr, m_tiles, depth;
};
static_assert(offsetof(BatchParams, y) == kPreloadWords * 4, "y starts the part that is not preloaded");

// BITS: 4 or 8.  GROUP: 64 or 32.
constexpr int batch_x_bytes(int mr, int bits) { return mr * 4 * (128 * 8 / bits) * 2; }
// DEPTH of one: x of a chunk comes in pieces, of 64 values a row above 16 rows, of at most 4 KB below.  Two and more, where a
// workgroup has a CU to itself: pieces that many times as long, or, where a chunk is one piece, that many chunks in flight.
constexpr int batch_x_piece1(int mr, int bits)
{
  return mr >= 8 ? mr * 512 : batch_x_bytes(mr, bits) < 4096 ? batch_x_bytes(mr, bits) : 4096;
}
constexpr int batch_ring(int mr, int bits, int depth) { return batch_x_piece1(mr, bits) == batch_x_bytes(mr, bits) ? depth : 1; }
constexpr int batch_x_piece(int mr, int bits, int depth)
{
  return batch_x_piece1(mr, bits) * (depth / batch_ring(mr, bits, depth));
}
constexpr int batch_slot_bytes(int t, int mr, int bits, int depth) { return t * 2048 + batch_x_piece(mr, bits, depth); }

template <int T, int MR, int BITS, int GROUP, int DEPTH>
struct BatchShape {
  static constexpr int CK = 128 * 8 / BITS;                       // values of K per chunk
  static constexpr int AT = MR >= 8 ? MR / 4 : 1;                 // MFMA tiles of 16 rows of x
  static constexpr int RA = MR >= 8 ? 4 : MR;                     // accumulator registers of one
  static constexpr int XS = batch_x_bytes(MR, BITS) / batch_x_piece(MR, BITS, DEPTH);   // pieces of x per chunk
  static constexpr int RING = batch_ring(MR, BITS, DEPTH);        // slots of a wavefront (one where XS > 1)
  static constexpr int SK = CK / XS;                              // values of K per piece
  static constexpr int XROWB = SK * 2;
  static constexpr int XLOADS = MR * 4 * XROWB / 1024;            // direct-to-LDS loads per piece
  static constexpr int CLOADS = T * 2;                            // ... and per chunk of codes
  static constexpr int SLOT = (CLOADS + XLOADS) * 1024;
  static constexpr int SG = CK / GROUP;                           // groups per chunk
  static constexpr int SGW = SG / 2;                              // their scales of one row, in words
  static constexpr int MPG = GROUP / 32;                          // MFMAs per group
  static_assert(RING == 1 || XS == 1, "");
  static_assert(T * AT * RA * kWave * 4 <= RING * SLOT, "the partial results lie over the slots");
};

// Whether two workgroups may share a CU: at most 128 registers per lane (the build refuses a spill).
constexpr bool batch_two_per_cu(int t, int mr, int group, int depth)
{
  return depth == 1 && t <= 2 && mr <= 8 && !(t == 2 && group == 32 && mr == 8);
}

inline int batch_scale_bytes(int tiles, int K, int group) { return (tiles * 16 * (K / group) * 2 + 1023) / 1024 * 1024; }

namespace {

template <bool F16>
__device__ __forceinline__ floatx4 batch_mfma(u32x4 a, u32x4 b, floatx4 c)
{
  if constexpr (F16) {
    typedef _Float16 halfx8 __attribute__((ext_vector_type(8)));
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(halfx8, a), __builtin_bit_cast(halfx8, b), c, 0, 0, 0);
  } else {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c, 0, 0, 0);
  }
}

// Eight nibbles of a word -> eight elements q, in order.  A byte 0..15 read as fp8 (E4M3) is q * 2^-9 (exponent fields 0
// and 1 are one linear range), so the scaled conversion by 2^9 gives q, two a time.
template <bool F16>
__device__ __forceinline__ u32x4 batch_nibbles(uint32_t word, uint32_t mask)
{
  const uint32_t even = word & mask, odd = (word >> 4) & mask;
  const uint32_t lo = __builtin_amdgcn_perm(odd, even, 0x05010400u), hi = __builtin_amdgcn_perm(odd, even, 0x07030602u);
  u32x4 v;
  if constexpr (F16) {
    v[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 512.0f, false));
    v[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(lo, 512.0f, true));
    v[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 512.0f, false));
    v[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_f16_fp8(hi, 512.0f, true));
  } else {
    v[0] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, false));
    v[1] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(lo, 512.0f, true));
    v[2] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, false));
    v[3] = __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(hi, 512.0f, true));
  }
  return v;
}

// Eight bytes of two words -> eight bf16 values q, in order (0..255 has at most eight significant bits: the upper
// half of the fp32 value is exact).
__device__ __forceinline__ u32x4 batch_bytes(uint32_t w0, uint32_t w1)
{
  auto pair = [](uint32_t lo, uint32_t hi) {
    return __builtin_amdgcn_perm(__float_as_uint((float)hi), __float_as_uint((float)lo), 0x07060302u);
  };
  u32x4 v;
  v[0] = pair(w0 & 0xffu, (w0 >> 8) & 0xffu);
  v[1] = pair((w0 >> 16) & 0xffu, w0 >> 24);
  v[2] = pair(w1 & 0xffu, (w1 >> 8) & 0xffu);
  v[3] = pair((w1 >> 16) & 0xffu, w1 >> 24);
  return v;
}

// 16 bytes per lane, global (base + off) -> LDS at lds_dst + 16 * lane.  Written out by hand: the compiler waits for every
// such load that it knows about before any later LDS read, whatever the load fills.  The LDS base travels in M0, bound as an
// operand (the s_nop is the wait state between that write and the load).
__device__ __forceinline__ void batch_to_lds(const uint8_t* base, uint32_t off, void* lds_dst)
{
  const uint32_t dst = (uint32_t)(uintptr_t)(__attribute__((address_space(3))) uint8_t*)(uint8_t*)lds_dst;
  const uint32_t m0v = __builtin_amdgcn_readfirstlane(dst);
  asm volatile("s_nop 0\n\tglobal_load_lds_dwordx4 %0, %1" : : "v"(off), "s"(base), "{m0}"(m0v) : "memory");
}

}  // namespace

// MR: accumulator registers per lane and tile, 1 / 2 / 4 / 8 / 12 / 16 for up to 4 / 8 / 16 / 32 / 48 / 64 rows
// of x.  Row m of an MFMA
// tile of x sits in MFMA row 4*(m%4) + m/4, so that output row m is register m/4 of lane group m%4 and up to four rows
// need one register.
template <int T, int MR, int BITS, int GROUP, bool F16, bool SONLY, int DEPTH>
__global__ __launch_bounds__(kBatchWaves * 64, batch_two_per_cu(T, MR, GROUP, DEPTH) ? 4 : 2) void
qmv_batch_kernel(VPQ_PRELOADED_WORDS, const PreloadTail<BatchParams> tail)
{
  using S = BatchShape<T, MR, BITS, GROUP, DEPTH>;
  const BatchParams p = preload_assemble<BatchParams>(VPQ_PRELOADED_WORD_LIST, tail);
  extern __shared__ __attribute__((aligned(16))) uint8_t lds[];

  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6);
  const int fr = lane & 15;                 // MFMA row (A) / column (B, D) of this lane
  const int g = lane >> 4;                  // k sub-block of this lane

  // Workgroups go to the XCDs round robin: the workgroups of one block of weight rows (one per tile of rows of x) are
  // eight apart, so that the second reads the codes from its XCD's L2.
  int nb = blockIdx.x, mt = 0;
  if (p.m_tiles > 1) {
    const int span = 8 * p.m_tiles;
    const int q = nb / span, r = nb - q * span;
    nb = q * 8 + (r & 7);
    mt = r >> 3;
  }
  if (nb >= p.blocks) { return; }
  const int m0 = mt * p.rows;
  const int rows = (p.M - m0) < p.rows ? (p.M - m0) : p.rows;
  if (rows <= 0) { return; }

  const uint32_t* w_ = p.w;
  const uint16_t* scales_ = p.scales;
  const uint16_t* biases_ = p.biases;
  void* y_ = p.y;
  int N_ = p.N;
  if (p.nseg > 1 && nb >= p.seg_first[0]) {                 // (constant indexes: a variable one would put p into scratch)
    int first = p.seg_first[0];
    QmvSeg seg = p.seg[0];
    if (p.nseg > 2 && nb >= p.seg_first[1]) { first = p.seg_first[1]; seg = p.seg[1]; }
    if (p.nseg > 3 && nb >= p.seg_first[2]) { first = p.seg_first[2]; seg = p.seg[2]; }
    w_ = seg.w; scales_ = seg.scales; biases_ = seg.biases; y_ = seg.y; N_ = seg.N;
    nb -= first;
  }
  const int n0 = nb * (T * 16);
  const int n_live = (N_ - n0) < T * 16 ? (N_ - n0) : T * 16;
  const int Kg = p.K / GROUP;
  const uint32_t row_bytes = (uint32_t)p.K * BITS / 8;
  const int chunks = (p.K + S::CK - 1) / S::CK;

  uint8_t* const slots = lds + wave * (S::RING * S::SLOT);
  uint8_t* slot = slots;                                    // of the chunk in hand
  uint8_t* sblk = lds + kBatchWaves * S::RING * S::SLOT;
  const int sb_bytes = n_live * Kg * 2;
  const int sb_loads = (sb_bytes + 1023) >> 10;
  uint8_t* bblk = sblk + sb_loads * 1024;

  // ---- requests ----
  const uint8_t* wtile = reinterpret_cast<const uint8_t*>(w_) + (size_t)n0 * row_bytes;
  const uint8_t* xtile = reinterpret_cast<const uint8_t*>(p.x) + (size_t)m0 * p.K * 2;
  // Load i of a chunk's codes covers rows 8i..8i+7: lane l takes row 8i + l/8, LDS piece l%8 of its 128 bytes; the
  // swizzle key (row/2)%8 is l/16 with bit 2 flipped in every second load.  A load's offset is one v_xad from two
  // registers (kept opaque, or the compiler would hold one register per load over the loop); rows past the last one
  // repeat it.
  uint32_t code_piece = (uint32_t)(((lane & 7) ^ (lane >> 4)) * 16);
  uint32_t code_row = __umul24((uint32_t)(lane >> 3), row_bytes);
  auto request_codes = [&](int c, uint8_t* to) {
    const uint8_t* base = wtile + (size_t)c * 128;
    const int left = (int)row_bytes - c * 128;              // bytes of a row from here on
    uint32_t rb = row_bytes;
    asm volatile("" : "+v"(code_piece), "+s"(rb));
    if (left >= 128 && n_live == T * 16) {
#pragma unroll
      for (int i = 0; i < S::CLOADS; ++i) {
        batch_to_lds(base, (code_piece ^ ((i & 1) * 64)) + code_row, to + i * 1024);
        base += 8 * (size_t)rb;
      }
    } else {
#pragma unroll
      for (int i = 0; i < S::CLOADS; ++i) {
        const int row = i * 8 + (lane >> 3);
        const uint32_t at = code_piece ^ ((i & 1) * 64);
        batch_to_lds(base, __umul24((uint32_t)(row < n_live ? row : n_live - 1), rb) + ((int)at < left ? at : 0),
                     to + i * 1024);
      }
    }
  };
  // Lane l of load i of x takes 16 bytes of row (i*1024 + l*16) / XROWB; swizzle key row % 16
  // ((row/2) % 8 in rows of 128 bytes).  Rows past the live ones
  // are not staged: their MFMA rows are computed from what the slot holds and not stored.
  constexpr int kXPieces = S::XROWB / 16, kRowsPerLoad = 1024 / S::XROWB;
  const uint32_t x_bytes = (uint32_t)p.K * 2u;
  uint32_t x_piece = (uint32_t)(((lane & (kXPieces - 1)) ^ (kXPieces >= 16 ? lane / kXPieces : lane >> 4)) * 16);
  uint32_t x_row = __umul24((uint32_t)(lane / kXPieces), x_bytes);
  auto request_x = [&](int c, int sub, uint8_t* to) {
    const int k0 = c * S::CK + sub * S::SK;
    const int left = (p.K - k0) * 2;
    const uint8_t* base = xtile + (size_t)k0 * 2;
    uint32_t xb = x_bytes;
    int live = rows;
    asm volatile("" : "+v"(x_piece), "+s"(xb));
    if constexpr (S::XLOADS > 4) { asm volatile("" : "+s"(live)); }   // (no comparison per load is held over the loop)
#pragma unroll
    for (int i = 0; i < S::XLOADS; ++i) {
      const uint32_t at = x_piece ^ (uint32_t)(kXPieces >= 16 ? ((i * kRowsPerLoad) & 15) * 16 : (i & 1) * 64);
      if (left >= S::XROWB && (i + 1) * kRowsPerLoad <= live) {
        batch_to_lds(base, at + x_row, to + (S::CLOADS + i) * 1024);
      } else if (i * kRowsPerLoad < live) {
        int row = lane / kXPieces;
        asm volatile("" : "+v"(row));                       // (the rare path: nothing of it is held over the loop)
        const int last = live - 1 - i * kRowsPerLoad;
        batch_to_lds(base, __umul24((uint32_t)(row < last ? row : last), xb) + ((int)at < left ? at : 0),
                     to + (S::CLOADS + i) * 1024);
      }
      base += kRowsPerLoad * (size_t)xb;
    }
  };
  // One block of scales (biases): whole 16-byte pieces here, a last partial piece after the wait below.
  auto request_block = [&](const uint16_t* src, uint8_t* dst) {
    const int last = (sb_bytes >> 4) - 1;
    if (last >= 0) {
      for (int i = wave; i < sb_loads; i += kBatchWaves) {
        int piece = i * 64 + lane;
        if (piece > last) { piece = last; }
        batch_to_lds(reinterpret_cast<const uint8_t*>(src), (uint32_t)piece * 16, dst + i * 1024);
      }
    }
  };
  const uint16_t* sc_src = scales_ + (size_t)n0 * Kg;
  const uint16_t* bi_src = SONLY ? nullptr : biases_ + (size_t)n0 * Kg;
  request_block(sc_src, sblk);
  if (!SONLY) { request_block(bi_src, bblk); }
  const int mine = wave < chunks ? (chunks - wave + kBatchWaves - 1) / kBatchWaves : 0;   // chunks of this wavefront
#pragma unroll
  for (int i = 0; i < S::RING; ++i) {
    if (i < mine) {
      request_x(wave + i * kBatchWaves, 0, slots + i * S::SLOT);
      request_codes(wave + i * kBatchWaves, slots + i * S::SLOT);
    }
  }
  // the scales: older than every chunk's loads (of x at least one each)
  if (S::RING > 1 && mine >= S::RING) {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(S::RING * (S::CLOADS + 1) - 1) : "memory");
  } else if (mine > 0) {
    asm volatile("s_waitcnt vmcnt(%0)" : : "n"(S::CLOADS) : "memory");
  } else {
    asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
  }
  asm volatile("s_barrier" : : : "memory");                 // (__syncthreads would wait for the chunks as well)
  // The arguments that only the store needs are read by here, behind the requests and not when it waits for them.
  asm volatile("" : : "s"(y_), "s"(p.residual), "s"(p.gate_act), "s"(p.y_f32));
  if ((sb_bytes & 15) != 0) {                               // the last rows of an N that is not a multiple of 8
    const int at = (sb_bytes >> 4) * 8 + (int)threadIdx.x;
    if (at < (sb_bytes >> 1)) {
      reinterpret_cast<uint16_t*>(sblk)[at] = sc_src[at];
      if (!SONLY) { reinterpret_cast<uint16_t*>(bblk)[at] = bi_src[at]; }
    }
    __syncthreads();
  }

  uint32_t mask = 0x0f0f0f0fu;
  asm volatile("" : "+s"(mask));                            // no instruction: only hides the constant from folding
  // What x is contracted with for sum(x) of a group: the negated middle code (4 bits), or one.
  u32x4 unit;
  unit[0] = unit[1] = unit[2] = unit[3] = BITS == 8 ? 0x3f803f80u : F16 ? 0xc800c800u : 0xc100c100u;
  asm volatile("" : "+v"(unit));

  // One rounding a 64 values of K in the long sum.  Groups of 64: acc sums scale * sum(x (q - middle)), off the offsets
  // (bias + middle * scale) * sum(x), small for packs whose zero points lie near the middle code.  Groups of 32: off
  // holds the first of two groups.
  float acc[T][S::AT][S::RA], off[T][S::AT][S::RA];
#pragma unroll
  for (int t = 0; t < T; ++t) {
#pragma unroll
    for (int a = 0; a < S::AT; ++a) {
#pragma unroll
      for (int q = 0; q < S::RA; ++q) { acc[t][a][q] = off[t][a][q] = 0.0f; }
    }
  }

  // A lane's operands of a chunk.  MFMA j takes from lane (fr, g) the eight values at k = 32j + 8g (groups of 32) or
  // at k = 64(j/2) + 16g + 8(j%2) (groups of 64): any order inside a group is right as long as codes and x agree.
  constexpr int kPieceMfmas = S::SK / 32;
  uint32_t cw[T][8];
  u32x4 xq[S::AT][kPieceMfmas];
  uint32_t sw[T][S::SGW], bw[T][S::SGW];

  auto take_codes = [&](int c) {
#pragma unroll
    for (int t = 0; t < T; ++t) {
      const int row = t * 16 + fr;
      const uint8_t* rp = slot + row * 128;
      const int key = (row >> 1) & 7;
      if constexpr (BITS == 4 && GROUP == 64) {
#pragma unroll
        for (int grp = 0; grp < 4; ++grp) {
          const u32x2 v = *reinterpret_cast<const u32x2*>(rp + (((2 * grp + (g >> 1)) ^ key) * 16) + (g & 1) * 8);
          cw[t][2 * grp] = v[0];
          cw[t][2 * grp + 1] = v[1];
        }
      } else if constexpr (BITS == 4) {
#pragma unroll
        for (int j = 0; j < 8; ++j) { cw[t][j] = *reinterpret_cast<const uint32_t*>(rp + ((j ^ key) * 16) + g * 4); }
      } else if constexpr (GROUP == 64) {
#pragma unroll
        for (int grp = 0; grp < 2; ++grp) {
          const u32x4 v = *reinterpret_cast<const u32x4*>(rp + (((4 * grp + g) ^ key) * 16));
#pragma unroll
          for (int i = 0; i < 4; ++i) { cw[t][4 * grp + i] = v[i]; }
        }
      } else {
#pragma unroll
        for (int j = 0; j < 4; ++j) {
          const u32x2 v = *reinterpret_cast<const u32x2*>(rp + (((2 * j + (g >> 1)) ^ key) * 16) + (g & 1) * 8);
          cw[t][2 * j] = v[0];
          cw[t][2 * j + 1] = v[1];
        }
      }
      // scales and biases of the chunk's groups (past the row's end: neighbours, never used)
      const int at = row * Kg + c * S::SG;
      const uint16_t* sp = reinterpret_cast<const uint16_t*>(sblk) + at;
      const uint16_t* bp = reinterpret_cast<const uint16_t*>(bblk) + at;
      if ((Kg & (S::SG - 1)) == 0) {
        __builtin_memcpy(sw[t], __builtin_assume_aligned(sp, S::SG * 2), S::SG * 2);
        if (!SONLY) { __builtin_memcpy(bw[t], __builtin_assume_aligned(bp, S::SG * 2), S::SG * 2); }
      } else {
#pragma unroll
        for (int i = 0; i < S::SGW; ++i) {
          sw[t][i] = (uint32_t)sp[2 * i] | ((uint32_t)sp[2 * i + 1] << 16);
          if (!SONLY) { bw[t][i] = (uint32_t)bp[2 * i] | ((uint32_t)bp[2 * i + 1] << 16); }
        }
      }
    }
  };
  auto take_x = [&]() {
#pragma unroll
    for (int a = 0; a < S::AT; ++a) {
      const int m_real = a * 16 + 4 * (fr & 3) + (fr >> 2);
      const int row = m_real < MR * 4 ? m_real : MR * 4 - 1;   // (MFMA rows past the slot's repeat its last)
      const uint8_t* rp = slot + S::CLOADS * 1024 + row * S::XROWB;
      const int key = kXPieces >= 16 ? row & 15 : (row >> 1) & 7;
#pragma unroll
      for (int j = 0; j < kPieceMfmas; ++j) {
        // (the upper bits of the piece are above the key: an offset instead of another address)
        const int piece = GROUP == 64 ? 8 * (j >> 1) + 2 * g + (j & 1) : 4 * j + g;
        xq[a][j] = *reinterpret_cast<const u32x4*>(rp + (((piece & 15) ^ key) * 16) + (j >> 2) * 256);
      }
    }
  };

  // Contracts piece `sub` of the taken chunk; PART: only its first `live` groups are inside K.
  auto contract_as = [&](auto sub_c, auto part_c, int live) {
    constexpr int kGroups = S::SK / GROUP, kG0 = decltype(sub_c)::value * kGroups;
#pragma unroll
    for (int grp = 0; grp < kGroups; ++grp) {
      if (decltype(part_c)::value && grp >= live) { break; }
      floatx4 xs[S::AT];
#pragma unroll
      for (int a = 0; a < S::AT; ++a) {
        xs[a] = floatx4{0.f, 0.f, 0.f, 0.f};
#pragma unroll
        for (int j = 0; j < S::MPG; ++j) { xs[a] = batch_mfma<F16>(xq[a][grp * S::MPG + j], unit, xs[a]); }
      }
      const int gc = kG0 + grp;                              // group of the chunk
#pragma unroll
      for (int t = 0; t < T; ++t) {
        floatx4 s4[S::AT];
#pragma unroll
        for (int a = 0; a < S::AT; ++a) { s4[a] = BITS == 4 ? xs[a] : floatx4{0.f, 0.f, 0.f, 0.f}; }
#pragma unroll
        for (int j = 0; j < S::MPG; ++j) {
          const int jc = gc * S::MPG + j;                    // MFMA of the chunk
          u32x4 b;
          if constexpr (BITS == 4) {
            b = batch_nibbles<F16>(cw[t][jc], mask);
          } else {
            b = batch_bytes(cw[t][2 * jc], cw[t][2 * jc + 1]);
          }
#pragma unroll
          for (int a = 0; a < S::AT; ++a) { s4[a] = batch_mfma<F16>(xq[a][grp * S::MPG + j], b, s4[a]); }
        }
        const float s = (gc & 1) ? elt_hi_to_f32<F16>(sw[t][gc >> 1]) : elt_lo_to_f32<F16>(sw[t][gc >> 1]);
        float b2 = 0.0f;                                     // (bias + 8 scale) / -8; 8 bits: the bias
        if constexpr (!SONLY) {
          b2 = (gc & 1) ? elt_hi_to_f32<F16>(bw[t][gc >> 1]) : elt_lo_to_f32<F16>(bw[t][gc >> 1]);
          if (BITS == 4) { b2 = fmaf(b2, -0.125f, -s); }
        }
#pragma unroll
        for (int a = 0; a < S::AT; ++a) {
#pragma unroll
          for (int q = 0; q < S::RA; ++q) {
            if constexpr (BITS == 8) {
              acc[t][a][q] = fmaf(s, s4[a][q], acc[t][a][q]);
              acc[t][a][q] = fmaf(b2, xs[a][q], acc[t][a][q]);
            } else if constexpr (GROUP == 64) {
              acc[t][a][q] = fmaf(s, s4[a][q], acc[t][a][q]);
              off[t][a][q] = fmaf(b2, xs[a][q], off[t][a][q]);
            } else {
              // (not contracted: the product of a last, single group would join its addition without the bias between them, and
              // a Q4_0 pack not have the bits of one that stores its biases)
#pragma clang fp contract(off)
              float v = (grp & 1) == 0 ? s * s4[a][q] : fmaf(s, s4[a][q], off[t][a][q]);
              if (!SONLY) { v = fmaf(b2, xs[a][q], v); }
              if ((grp & 1) == 0 && !(decltype(part_c)::value && grp + 1 >= live)) {
                off[t][a][q] = v;
              } else {
                acc[t][a][q] += v;
              }
            }
          }
        }
      }
    }
  };
  auto contract = [&](auto sub_c, int live) {
    if (live >= S::SK / GROUP) {
      contract_as(sub_c, std::false_type(), live);
    } else {
      contract_as(sub_c, std::true_type(), live);
    }
  };

  // The next chunk's codes are requested behind the piece of x after which they have the longest time that does not
  // make a later piece wait for them (loads return in order).
  constexpr int kCodesAt = S::XS >= 2 ? S::XS - 2 : 0;
  if constexpr (S::RING > 1) {
    // Loads return in order: a chunk is there when no more are out than the chunks behind it have.
    const int x_loads = (rows + kRowsPerLoad - 1) / kRowsPerLoad;
    auto arrive = [&](int behind) {
      auto wait = [&](auto x_c) {
        constexpr int kLoads = S::CLOADS + decltype(x_c)::value;
        if (S::RING > 2 && behind >= 2) {
          asm volatile("s_waitcnt vmcnt(%0)" : : "n"(2 * kLoads) : "memory");
        } else if (behind >= 1) {
          asm volatile("s_waitcnt vmcnt(%0)" : : "n"(kLoads) : "memory");
        } else {
          asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
        }
      };
      if (S::XLOADS > 3 && x_loads > 3) {
        wait(std::integral_constant<int, 4>());
      } else if (S::XLOADS > 2 && x_loads == 3) {
        wait(std::integral_constant<int, 3>());
      } else if (S::XLOADS > 1 && x_loads == 2) {
        wait(std::integral_constant<int, 2>());
      } else {
        wait(std::integral_constant<int, 1>());
      }
    };
    static_assert(S::XLOADS <= 4, "");
    for (int i = 0; i < mine; ++i) {
      const int c = wave + i * kBatchWaves, behind = mine - 1 - i;
      arrive(behind < S::RING - 1 ? behind : S::RING - 1);
      take_codes(c);
      take_x();
      asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
      if (i + S::RING < mine) {
        request_x(c + S::RING * kBatchWaves, 0, slot);
        request_codes(c + S::RING * kBatchWaves, slot);
      }
      contract(std::integral_constant<int, 0>(), (p.K - c * S::CK) / GROUP);
      slot = slot == slots + (S::RING - 1) * S::SLOT ? slots : slot + S::SLOT;
    }
  } else
  for (int c = wave; c < chunks; c += kBatchWaves) {
    const int nxt = c + kBatchWaves;
    const bool more = nxt < chunks;                          // (a chunk that ends past K is its wavefront's last)
    auto piece = [&](auto s_c) {
      constexpr int s = decltype(s_c)::value;
      const int left = p.K - c * S::CK - s * S::SK;
      if (s > 0 && left <= 0) { return; }
      if (s > 0 && s == kCodesAt + 1 && more) {
        asm volatile("s_waitcnt vmcnt(%0)" : : "n"(S::CLOADS) : "memory");
      } else {
        asm volatile("s_waitcnt vmcnt(0)" : : : "memory");
      }
      if (s == 0) { take_codes(c); }
      take_x();
      asm volatile("s_waitcnt lgkmcnt(0)" : : : "memory");
      if (s + 1 < S::XS) {
        if (left > S::SK) { request_x(c, s + 1, slot); }
      } else if (more) {
        request_x(nxt, 0, slot);
      }
      if (s == kCodesAt && more) { request_codes(nxt, slot); }
      contract(s_c, left / GROUP);
    };
    piece(std::integral_constant<int, 0>());
    if constexpr (S::XS > 1) { piece(std::integral_constant<int, 1>()); }
    if constexpr (S::XS > 2) {
      piece(std::integral_constant<int, 2>());
      piece(std::integral_constant<int, 3>());
    }
  }
  __syncthreads();

  // ---- the wavefronts' partial results: sums[tile][a][register][wave][lane], over the slots ----
  float* sums = reinterpret_cast<float*>(lds);
#pragma unroll
  for (int t = 0; t < T; ++t) {
#pragma unroll
    for (int a = 0; a < S::AT; ++a) {
#pragma unroll
      for (int q = 0; q < S::RA; ++q) {
        sums[(((t * S::AT + a) * S::RA + q) * kBatchWaves + wave) * kWave + lane] =
            BITS == 4 && GROUP == 64 ? acc[t][a][q] + off[t][a][q] : acc[t][a][q];
      }
    }
  }
  if constexpr (T * S::AT * S::RA <= 16) {
    // (few: spread over all wavefronts.  As quads 4096 -> 4096 at 16 rows takes 6.9 us for 6.2; more as these 31.0 for 30.5 of
    // 4096 -> 24576 at 48 rows.)
    // Wavefront w adds up and stores rows r = w, w + 8, ... of sums (r = (t * AT + a) * RA + q).
    constexpr int kOuts = T * S::AT * S::RA, kOutsPer = (kOuts + kBatchWaves - 1) / kBatchWaves;
    auto out_m = [&](int r) { return (r / S::RA) % S::AT * 16 + 4 * (r % S::RA) + g; };
    auto out_n = [&](int r) { return r / (S::RA * S::AT) * 16 + fr; };
    // (the residual is on its way while the wavefronts meet)
    uint16_t res[kOutsPer];
    if (p.residual != nullptr && p.gate_act == 0) {
#pragma unroll
      for (int i = 0; i < kOutsPer; ++i) {
        const int r = wave + i * kBatchWaves, m = out_m(r), n = out_n(r);
        res[i] = r < kOuts && m < rows && n < n_live ? p.residual[(size_t)(m0 + m) * N_ + n0 + n] : 0;
      }
    }
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");   // (__syncthreads would wait for the residual as well)
    float totals[kOutsPer];
#pragma unroll
    for (int i = 0; i < kOutsPer; ++i) {
      const int r = wave + i * kBatchWaves;
      const float* sp = sums + (r < kOuts ? r : 0) * (kBatchWaves * kWave) + lane;
      float part[kBatchWaves];
#pragma unroll
      for (int wv = 0; wv < kBatchWaves; ++wv) { part[wv] = sp[wv * kWave]; }
      totals[i] = 0.0f;
#pragma unroll
      for (int wv = 0; wv < kBatchWaves; ++wv) { totals[i] += part[wv]; }     // (wavefronts without a chunk add +0)
    }
#pragma unroll
    for (int i = 0; i < kOutsPer; ++i) {
      const int r = wave + i * kBatchWaves;
      if (r >= kOuts) { break; }
      float total = totals[i];
      const int m_loc = out_m(r), n_loc = out_n(r);
      const bool ok = m_loc < rows && n_loc < n_live;
      const int m = m0 + m_loc, n = n0 + n_loc;
      unsigned long long bad = __ballot(ok && (__float_as_uint(total) & 0x7f800000u) == 0x7f800000u);
      while (bad != 0) {                                       // one output of the wavefront at a time, all lanes on it
        const int src = __builtin_ctzll(bad);
        bad &= bad - 1;
        const int row = __builtin_amdgcn_readlane(n_loc, src), mb = __builtin_amdgcn_readlane(m, src);
        const float plain = plain_sum<BITS, GROUP, F16, SONLY>(
            wtile + (size_t)row * row_bytes, sc_src + (size_t)row * Kg, SONLY ? nullptr : bi_src + (size_t)row * Kg,
            p.x + (size_t)mb * p.K, p.K);
        if (lane == src) { total = plain; }
      }
      if (p.gate_act) {
        // Lanes 2j and 2j+1 hold the gate and the up sum of one feature (N is even).
        const float up = from_neighbour_lane(total);
        if (ok && (lane & 1) == 0) {
          const float v = gated_f32(p.gate_act, total, up);
          const size_t o = (size_t)m * (N_ >> 1) + (n >> 1);
          if (p.y_f32) {
            reinterpret_cast<float*>(y_)[o] = v;
          } else {
            reinterpret_cast<uint16_t*>(y_)[o] = (uint16_t)f32_to_elt_bits<F16>(v);
          }
        }
      } else if (ok) {
        const size_t o = (size_t)m * N_ + n;
        if (p.y_f32) {
          reinterpret_cast<float*>(y_)[o] = total;
        } else {
          uint32_t v = f32_to_elt_bits<F16>(total);
          if (p.residual != nullptr) {
            v = f32_to_elt_bits<F16>(elt_bits_to_f32<F16>(v) + elt_bits_to_f32<F16>(res[i]));
          }
          reinterpret_cast<uint16_t*>(y_)[o] = (uint16_t)v;
        }
      }
    }
  } else {
    // A thread adds up and stores quads of outputs, four weight rows of one row of x: quad i is lanes 4 (i % 16) .. + 3 of
    // register i / 16 = (t * AT + a) * RA + q.
    constexpr int kThreads = kBatchWaves * kWave, kQuads = T * S::AT * S::RA * 16, kRounds = (kQuads + kThreads - 1) / kThreads;
    const int tid = (int)threadIdx.x;
    auto quad_m = [](int i) { return (i >> 4) / S::RA % S::AT * 16 + 4 * ((i >> 4) % S::RA) + ((i >> 2) & 3); };
    auto quad_n = [](int i) { return (i >> 4) / (S::RA * S::AT) * 16 + (i & 3) * 4; };
    asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" : : : "memory");
#pragma unroll
    for (int j = 0; j < kRounds; ++j) {
      if (wave * kWave + j * kThreads >= kQuads) { break; }
      const bool on = tid + j * kThreads < kQuads;             // (all lanes stay: plain_sum needs them)
      const int i = on ? tid + j * kThreads : 0;
      floatx4 part[kBatchWaves], total = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
      for (int wv = 0; wv < kBatchWaves; ++wv) {
        part[wv] = *reinterpret_cast<const floatx4*>(sums + ((i >> 4) * kBatchWaves + wv) * kWave + (i & 15) * 4);
      }
#pragma unroll
      for (int wv = 0; wv < kBatchWaves; ++wv) { total += part[wv]; }         // (wavefronts without a chunk add +0)
      const int m_loc = quad_m(i), n_loc = quad_n(i), left = on && m_loc < rows ? n_live - n_loc : 0;
      const int m = m0 + m_loc, n = n0 + n_loc;
      unsigned bad_here = 0;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        if (e < left && (__float_as_uint(total[e]) & 0x7f800000u) == 0x7f800000u) { bad_here |= 1u << e; }
      }
      while (__ballot(bad_here != 0) != 0) {                   // one output of the wavefront at a time, all lanes on it
        const int src = __builtin_ctzll(__ballot(bad_here != 0));
        const int e = __builtin_ctz(__builtin_amdgcn_readlane((int)bad_here, src));
        const int row = __builtin_amdgcn_readlane(n_loc, src) + e, mb = __builtin_amdgcn_readlane(m, src);
        const float plain = plain_sum<BITS, GROUP, F16, SONLY>(
            wtile + (size_t)row * row_bytes, sc_src + (size_t)row * Kg, SONLY ? nullptr : bi_src + (size_t)row * Kg,
            p.x + (size_t)mb * p.K, p.K);
        if ((tid & 63) == src) {
          bad_here &= bad_here - 1;
#pragma unroll
          for (int f = 0; f < 4; ++f) { total[f] = f == e ? plain : total[f]; }
        }
      }
      if (left <= 0) {
      } else if (p.gate_act) {                                 // (gate, up, gate, up); N is even
        const float v0 = gated_f32(p.gate_act, total[0], total[1]);
        const float v1 = gated_f32(p.gate_act, total[2], total[3]);
        const size_t o = (size_t)m * (N_ >> 1) + (n >> 1);
        if (left > 2) {
          const uint32_t v = f32_to_elt_bits<F16>(v0) | f32_to_elt_bits<F16>(v1) << 16;
          __builtin_memcpy(reinterpret_cast<uint16_t*>(y_) + o, &v, 4);
        } else {
          reinterpret_cast<uint16_t*>(y_)[o] = (uint16_t)f32_to_elt_bits<F16>(v0);
        }
      } else {
        uint32_t v[4];
#pragma unroll
        for (int e = 0; e < 4; ++e) { v[e] = f32_to_elt_bits<F16>(total[e]); }
        uint16_t* yp = reinterpret_cast<uint16_t*>(y_) + (size_t)m * N_ + n;
        if (left >= 4) {
          const u32x2 w = {v[0] | v[1] << 16, v[2] | v[3] << 16};
          __builtin_memcpy(yp, &w, 8);
        } else {
          yp[0] = (uint16_t)v[0];
          if (left > 1) { yp[1] = (uint16_t)v[1]; }
          if (left > 2) { yp[2] = (uint16_t)v[2]; }
        }
      }
    }
  }
}

constexpr int kLdsOfCu = 160 * 1024;

// One instantiation's launch; the attribute is set once per kernel, whichever thread comes first (two may both set it,
// which is harmless; neither launches before its own call has returned).
template <int T, int MR, int BITS, int GROUP, bool F16, bool SONLY, int DEPTH>
hipError_t batch_launch_one(hipStream_t st, const BatchParams& p, size_t lds_bytes, int grid)
{
  static std::atomic<bool> ready{false};
  auto kern = qmv_batch_kernel<T, MR, BITS, GROUP, F16, SONLY, DEPTH>;
  if (!ready.load(std::memory_order_acquire)) {
    const hipError_t e = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                             hipFuncAttributeMaxDynamicSharedMemorySize, kLdsOfCu);
    if (e != hipSuccess) { return e; }
    ready.store(true, std::memory_order_release);
  }
  return launch_preloaded(kern, dim3((unsigned)grid), dim3(kBatchWaves * kWave), lds_bytes, st, p);
}

// The formats whose entrances end at 16 rows of x (binary16, 8 bits in groups of 32, Q4_0) have no forms for more.
template <int BITS, int GROUP, bool F16, bool SONLY = false>
hipError_t batch_launch(hipStream_t st, const BatchParams& p, const BatchPlan& plan, size_t lds_bytes, int grid)
{
#define VPQ_BATCH(T_, MR_, DEPTH_)                                                                    \
  if (plan.tiles == T_ && plan.mr == MR_ && plan.depth == DEPTH_) {                                   \
    return batch_launch_one<T_, MR_, BITS, GROUP, F16, SONLY, DEPTH_>(st, p, lds_bytes, grid);        \
  }
  constexpr bool kMoreRows = !F16 && !SONLY && !(BITS == 8 && GROUP == 32);
  VPQ_BATCH(1, 1, 1) VPQ_BATCH(1, 2, 1) VPQ_BATCH(1, 4, 1) VPQ_BATCH(2, 1, 1) VPQ_BATCH(2, 2, 1) VPQ_BATCH(2, 4, 1)
  VPQ_BATCH(1, 4, 2)
  if constexpr (BITS == 4) { VPQ_BATCH(2, 4, 2) }
  if constexpr (BITS == 8) { VPQ_BATCH(1, 1, 3) VPQ_BATCH(1, 2, 2) }
  if constexpr (kMoreRows) {
    VPQ_BATCH(1, 8, 1) VPQ_BATCH(2, 8, 1) VPQ_BATCH(2, 12, 1) VPQ_BATCH(2, 16, 1) VPQ_BATCH(3, 8, 1) VPQ_BATCH(3, 12, 1)
    if constexpr (BITS == 8) { VPQ_BATCH(1, 8, 2) VPQ_BATCH(2, 8, 2) }
  }
#undef VPQ_BATCH
  return hipErrorInvalidValue;
}

// The instantiations of the other formats (vpq_qmv_batch_twins.hip).
hipError_t launch_qmv_batch_twin(hipStream_t st, const BatchParams& p, const BatchPlan& plan, size_t lds_bytes, int grid,
                                 const BatchFormat& f);

}  // namespace vpq
