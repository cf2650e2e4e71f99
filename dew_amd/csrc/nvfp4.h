// The E2M1 codes of bf16 values under an NVFP4 block scale: the rule's own quotients, fl(fl(value / tensor) / each), rounded to
// nearest with ties to the even code, without a division and seven comparisons an element (thirty instructions; these are nine
// with the packing, and the launches are then bound by memory again).
//
// A quotient by a divisor known beforehand is a product with its correctly rounded reciprocal and one Newton step of two fused
// multiply-adds (P. Markstein, "Computation of elementary functions on the IBM RISC System/6000 processor", 1990): the IEEE
// quotient. Checked for every pair that comes here: values of eight significant bits over tensor scales fl(amax / 2688) of bf16
// amax, all 128 x 128 significands, and all 2^23 significands over the eight of e4m3. Tensor scales near the ends of fp32's range,
// where a step's remainder could be subnormal, keep the division; so do a weight held in fp32 and every operand that holds an
// infinity or a NaN, wherever it stands: the conversion instruction makes a NaN the largest code, where the comparisons read a
// zero, and a step from an infinity ends in inf - inf, a NaN. The instruction rounds as the rule does.
#pragma once

#include "common.h"

namespace dew {

// Whether an operand of this largest magnitude (a NaN where it holds one) and tensor scale takes the short form.
__device__ __forceinline__ bool nvfp4_in_range(float largest, float tensor) {
  return largest < __builtin_inff() && tensor >= 0x1p-80f && tensor <= 0x1p+117f;
}

// The reciprocal of a block's scale: 0 where the block has none (zeros, or a NaN), whose codes are all 0.
__device__ __forceinline__ float nvfp4_inverse(float each) { return each > 0.0f ? 1.0f / each : 0.0f; }

__device__ __forceinline__ float known_quotient(float value, float divisor, float inverse) {
  const float near = value * inverse;
  return fmaf(fmaf(-near, divisor, value), inverse, near);
}

// A tensor scale and a block's, each with its reciprocal.
struct Nvfp4Scales {
  float tensor, inverse_tensor, each, inverse_each;
  __device__ __forceinline__ float quotient(float value) const {
    const float magnitude = known_quotient(known_quotient(value, tensor, inverse_tensor), each, inverse_each);
    return copysignf(magnitude, value);  // (the step loses a zero's sign)
  }
  // Byte BYTE of `codes`: the codes of two values, the first in the low nibble (of a block that has a scale).
  template <int BYTE>
  __device__ __forceinline__ uint32_t pair(uint32_t codes, float first, float second) const {
    return __builtin_amdgcn_cvt_scalef32_pk_fp4_f32(codes, quotient(first), quotient(second), 1.0f, BYTE);
  }
  __device__ __forceinline__ uint32_t four(float a, float b, float c, float d) const {
    const uint32_t codes = pair<1>(pair<0>(0u, a, b), c, d);
    return inverse_each > 0.0f ? codes : 0u;
  }
  // Two values' codes times the block scale as bf16 patterns, the first below: exact (a code has two significant bits).
  __device__ __forceinline__ uint32_t values(float first, float second) const {
    typedef float f32x2_t __attribute__((ext_vector_type(2)));
    const f32x2_t value = __builtin_amdgcn_cvt_scalef32_pk_f32_fp4(pair<0>(0u, first, second), 1.0f, 0);
    const uint32_t both = __builtin_amdgcn_perm(__float_as_uint(value[1] * each), __float_as_uint(value[0] * each), 0x07060302u);
    return inverse_each > 0.0f ? both : 0u;
  }
};

// An operand's largest magnitude as fp32 bits (magnitudes order as their bit patterns do; a NaN's are the largest), from the `count` partial
// ones that a launch left, one a block: some hundred words for every wavefront that wants it, where one word would take a launch that clears
// it. In two parts, so that a wavefront's other loads go out between them: a lane's share, and the whole.
constexpr int kNvfp4Partials = 512;
__device__ __forceinline__ uint32_t nvfp4_share(const uint32_t* __restrict__ partials, int count) {
  uint32_t mine = 0;
  if (count == 1) return *partials;
#pragma unroll
  for (int i = 0; i < kNvfp4Partials / 64; ++i) mine = max(mine, partials[64 * i + threadIdx.x % 64]);
  return mine;
}
__device__ __forceinline__ float nvfp4_top(uint32_t mine) {
#pragma unroll
  for (int offset = 32; offset >= 1; offset >>= 1) mine = max(mine, static_cast<uint32_t>(__shfl_xor(static_cast<int>(mine), offset, 64)));
  return __uint_as_float(__builtin_amdgcn_readfirstlane(mine));
}

// largest / (6 * 448), fp32's least normal at least; 1 for an operand of zeros
__device__ __forceinline__ float nvfp4_tensor_scale(float top) { return top > 0.0f ? fmaxf(top / 2688.0f, 1.17549435e-38f) : 1.0f; }

// A block's scale: the least e4m3 at or above blockmax / tensor / 6, the nearest one and the next where that lies below.
__device__ __forceinline__ float nvfp4_block_scale(float block, float tensor) {
  const float ratio = (block / tensor) / 6.0f;
  uint32_t byte = __builtin_amdgcn_cvt_pk_fp8_f32(fminf(ratio, 448.0f), 0.0f, 0, false) & 0xFFu;
  if (__builtin_amdgcn_cvt_f32_fp8(byte, 0) < ratio) byte = min(byte + 1u, 0x7Eu);
  return __builtin_amdgcn_cvt_f32_fp8(byte, 0);
}

// The nearest E2M1 to a quotient by the block scale (ties to the even code) times that scale, without the quotient: for y = x / tensor and the block scale `each` (an e4m3
// value, four significant bits), fl(y / each) > t exactly where y > t each, and >= likewise, for each of the seven
// thresholds t (at most three significant bits, so t each is exact): a y above t each lies at least one ulp of t each
// above it, which is more than half an ulp of t above t in the quotient (their ratio is 1 / m or 2 / m for each's
// significand m < 2), so the quotient rounds past t; at or below, it cannot round above. One IEEE division an element
// instead of two.
__device__ __forceinline__ float e2m1_scaled(float magnitude, float each) {
  float value = magnitude > 0.25f * each ? 0.5f * each : 0.0f;
  value = magnitude >= 0.75f * each ? each : value;
  value = magnitude > 1.25f * each ? 1.5f * each : value;
  value = magnitude >= 1.75f * each ? 2.0f * each : value;
  value = magnitude > 2.5f * each ? 3.0f * each : value;
  value = magnitude >= 3.5f * each ? 4.0f * each : value;
  return magnitude > 5.0f * each ? 6.0f * each : value;
}

// Two values' codes times the block scale as bf16 patterns, the first below, by divisions: exact in bf16.
__device__ __forceinline__ uint32_t nvfp4_values_divided(float first, float second, float tensor, float each) {
  const float a = each > 0.0f ? first / tensor : 0.0f, b = each > 0.0f ? second / tensor : 0.0f;
  return (__float_as_uint(copysignf(e2m1_scaled(fabsf(a), each), a)) >> 16) | (__float_as_uint(copysignf(e2m1_scaled(fabsf(b), each), b)) & 0xFFFF0000u);
}

}  // namespace dew
