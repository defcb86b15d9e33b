// Codes of a weight tile -> the elements the GEMM kernels multiply: elt_rne(fp32(s * q + b)), the tile arithmetic of
// gpu-kernels/metal/quant/affine_qmm_steel.metal:78-96.
#pragma once

#include "vpq_device.h"

namespace vpq {

namespace {

// Byte I of a dword as fp32 (selects v_cvt_f32_ubyteI).
template <int I>
__device__ __forceinline__ float ubyte_f32(uint32_t v) { return (float)((v >> (8 * I)) & 0xffu); }

// 8 nibbles of one word -> 8 bf16 (F16: IEEE binary16) of fma(s, q, b), as one 16-byte LDS chunk.
template <bool F16 = false>
__device__ __forceinline__ uint4 dequant_word(uint32_t word, float s, float b)
{
  uint32_t lo = word & 0x0f0f0f0fu;                // q0 q2 q4 q6
  uint32_t hi = (word >> 4) & 0x0f0f0f0fu;         // q1 q3 q5 q7
  // No instruction: keeps the masked words as they are, so that each value is one v_cvt_f32_ubyteN
  // of them (otherwise the mask is folded into a bit-field extract per value, one instruction more).
  asm volatile("" : "+v"(lo), "+v"(hi));
  const float v0 = fmaf(s, ubyte_f32<0>(lo), b);
  const float v1 = fmaf(s, ubyte_f32<0>(hi), b);
  const float v2 = fmaf(s, ubyte_f32<1>(lo), b);
  const float v3 = fmaf(s, ubyte_f32<1>(hi), b);
  const float v4 = fmaf(s, ubyte_f32<2>(lo), b);
  const float v5 = fmaf(s, ubyte_f32<2>(hi), b);
  const float v6 = fmaf(s, ubyte_f32<3>(lo), b);
  const float v7 = fmaf(s, ubyte_f32<3>(hi), b);
  uint4 o;
  o.x = pack_elt2<F16>(v0, v1);
  o.y = pack_elt2<F16>(v2, v3);
  o.z = pack_elt2<F16>(v4, v5);
  o.w = pack_elt2<F16>(v6, v7);
  return o;
}

// The same values by fp8 conversions: a byte 0..15 read as E4M3 is q * 2^-9 (exponent fields 0 and 1 are one linear range),
// so the conversion scaled by 2^9 gives q exactly, two values an instruction.
template <bool F16 = false>
__device__ __forceinline__ uint4 dequant_word_fp8(uint32_t word, float s, float b)
{
  typedef float floatx2 __attribute__((ext_vector_type(2)));
  const uint32_t even = word & 0x0f0f0f0fu, odd = (word >> 4) & 0x0f0f0f0fu;
  const floatx2 e0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(even, 512.0f, false);
  const floatx2 e1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(even, 512.0f, true);
  const floatx2 o0 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(odd, 512.0f, false);
  const floatx2 o1 = __builtin_amdgcn_cvt_scalef32_pk_f32_fp8(odd, 512.0f, true);
  uint4 o;
  o.x = pack_elt2<F16>(fmaf(s, e0[0], b), fmaf(s, o0[0], b));
  o.y = pack_elt2<F16>(fmaf(s, e0[1], b), fmaf(s, o0[1], b));
  o.z = pack_elt2<F16>(fmaf(s, e1[0], b), fmaf(s, o1[0], b));
  o.w = pack_elt2<F16>(fmaf(s, e1[1], b), fmaf(s, o1[1], b));
  return o;
}

// 8 bytes of two packed words -> 8 bf16 of fma(s, q, b), as one 16-byte LDS chunk (the 8-bit pack).
__device__ __forceinline__ uint4 dequant_bytes(uint32_t w0, uint32_t w1, float s, float b)
{
  uint4 o;
  o.x = pack_bf16x2(fmaf(s, ubyte_f32<0>(w0), b), fmaf(s, ubyte_f32<1>(w0), b));
  o.y = pack_bf16x2(fmaf(s, ubyte_f32<2>(w0), b), fmaf(s, ubyte_f32<3>(w0), b));
  o.z = pack_bf16x2(fmaf(s, ubyte_f32<0>(w1), b), fmaf(s, ubyte_f32<1>(w1), b));
  o.w = pack_bf16x2(fmaf(s, ubyte_f32<2>(w1), b), fmaf(s, ubyte_f32<3>(w1), b));
  return o;
}

}  // namespace

}  // namespace vpq
