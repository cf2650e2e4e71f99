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

}  // namespace dew
