// The arithmetic of the BitLinear activation quantiser (BitLinearBitBLAS.activation_quant,
// examples/bitnet-1.58b/utils_quant.py:156-163), shared by the kernel of its own (dq_quant.hip) and the small-batch GEMM
// kernels that quantise their activations themselves:
//     s[m]   = (1 / max(max_k |x[m, k]|, 1e-5)) * 127      (fp32; what torch's `Qp / tensor` computes)
//     q[m,k] = clamp(round_half_even(float(x[m, k]) * s[m]), -128, 127)  -> int8
#pragma once

#include "dq_common.h"

namespace dq {

// Maximum over the 32 lanes of a half wave / over the wave; values are >= 0, so the zero fill of the moves is harmless.
__device__ __forceinline__ float half_wave_max(float v) {
  v = fmaxf(v, dpp_move<0xB1>(v));
  v = fmaxf(v, dpp_move<0x4E>(v));
  v = fmaxf(v, dpp_move<0x141>(v));
  v = fmaxf(v, dpp_move<0x140>(v));
  // all 16 lanes of a row hold the row maximum
  return fmaxf(v, __shfl_xor(v, 16));
}
__device__ __forceinline__ float wave_max(float v) {
  v = half_wave_max(v);
  return fmaxf(v, __shfl_xor(v, 32));
}

__device__ __forceinline__ float amax8(const half8_t& h, float amax) {
#pragma unroll
  for (int e = 0; e < 8; ++e) amax = fmaxf(amax, fabsf((float)h[e]));
  return amax;
}

// Qp / tensor in torch is tensor.reciprocal() * Qp: a correctly rounded reciprocal, then a product
__device__ __forceinline__ float act_scale(float amax) { return (1.0f / fmaxf(amax, 1e-5f)) * 127.f; }

// Eight activations -> eight int8.  Adding 1.5 * 2^23 rounds the product to the nearest whole number, ties to even, and
// leaves it in the low byte.  |x s| <= 127 (1 + 2^-22) whatever is finite, so of the clamp only the lower bound can act: on
// a NaN (of an infinity's zero scale, or in the input), which fmaxf takes to -128 as the clamp does.
__device__ __forceinline__ uint2_t quantise8(const half8_t& h, float s) {
#pragma clang fp contract(off)  // the product is rounded before the sum
  constexpr float kMagic = 12582912.f;
  uint32_t b[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x = (float)h[e] * s;
    const float y = x + kMagic;
    b[e] = __builtin_bit_cast(uint32_t, fmaxf(y, kMagic - 128.f));
  }
  uint2_t o;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t lo = __builtin_amdgcn_perm(b[4 * i + 1], b[4 * i], 0x0c0c0400u), hi = __builtin_amdgcn_perm(b[4 * i + 3], b[4 * i + 2], 0x04000c0cu);
    o[i] = lo | hi;
  }
  return o;
}

// The same for rows without infinities and NaN, whose largest magnitude is found in integers: 2 instructions an activation
// (and two more where one of the above is general) instead of 5.
typedef unsigned short ushort2_t __attribute__((ext_vector_type(2)));
constexpr uint32_t kLargestFinite = 0x7BFFu;  // bits of the largest finite fp16

// Bits of the largest magnitude of the even and of the odd elements, two at a time
__device__ __forceinline__ ushort2_t abits8(const half8_t& h, ushort2_t m) {
  const uint4_t d = __builtin_bit_cast(uint4_t, h);
#pragma unroll
  for (int i = 0; i < 4; ++i) m = __builtin_elementwise_max(m, __builtin_bit_cast(ushort2_t, d[i] & 0x7FFF7FFFu));
  return m;
}
__device__ __forceinline__ uint32_t half_wave_max_bits(ushort2_t m) {
  uint32_t v = max((uint32_t)m[0], (uint32_t)m[1]);
  v = max(v, dpp_move<0xB1>(v));
  v = max(v, dpp_move<0x4E>(v));
  v = max(v, dpp_move<0x141>(v));
  v = max(v, dpp_move<0x140>(v));
  return max(v, (uint32_t)__shfl_xor((int)v, 16));
}
__device__ __forceinline__ uint32_t wave_max_bits(ushort2_t m) {
  const uint32_t v = half_wave_max_bits(m);
  return max(v, (uint32_t)__shfl_xor((int)v, 32));
}
__device__ __forceinline__ float act_scale_of_bits(uint32_t bits) {
  return act_scale((float)__builtin_bit_cast(half_t, (unsigned short)bits));
}
__device__ __forceinline__ uint2_t quantise8_finite(const half8_t& h, float s) {
#pragma clang fp contract(off)  // the product is rounded before the sum
  uint32_t b[8];
#pragma unroll
  for (int e = 0; e < 8; ++e) {
    const float x = __builtin_fmaf((float)h[e], s, 0.f);  // a product (but for the sign of a zero) that takes its operand in fp16
    const float y = x + 12582912.f;
    b[e] = __builtin_bit_cast(uint32_t, y);
  }
  uint2_t o;
#pragma unroll
  for (int i = 0; i < 2; ++i) {
    const uint32_t lo = __builtin_amdgcn_perm(b[4 * i + 1], b[4 * i], 0x0c0c0400u), hi = __builtin_amdgcn_perm(b[4 * i + 3], b[4 * i + 2], 0x0c0c0400u);
    o[i] = __builtin_amdgcn_perm(hi, lo, 0x05040100u);
  }
  return o;
}

}  // namespace dq
