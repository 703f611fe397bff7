// Arithmetic of the eager attention's softmax (PE_ATTN_EAGER), the reference's
// rounding of a score and of its exponential (src/pe/nn.py:84-87). Host and
// device: tests/test_eager_arithmetic.py sweeps these functions on the CPU.
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/pe_hip.h"

// The fp32 quotient x / sqrt(128) (torch divides in fp32) of a value x of the
// 16-bit type, exact enough that rounding it to that type gives what the
// correctly rounded quotient gives, for all 65536 values of x: infinities, the
// sign of zero and NaN among them. bf16 needs the product with the reciprocal
// alone; fp16 the reciprocal in two parts, both positive, so that an infinite
// score (a product past 65504) stays the infinity that it is: the remainder
// step of a division would subtract infinities.
template <int DT>
__host__ __device__ __forceinline__ float eager_quotient(float x) {
  constexpr float kInvHi = 0x1.6a09e6p-4f, kInvLo = 0x1.9fcef4p-29f;  // 1 / float(sqrt(128))
  if constexpr (DT == PE_DTYPE_F16) return fmaf(x, kInvHi, x * kInvLo);
  return x * kInvHi;
}

// exp(x) for x <= 0: 2^(x log2 e), the product's rounding error put back to
// first order, so that the result is as exact as v_exp_f32. Far below 2^-149
// the argument is held at a finite value whose exponential is 0 (the error
// term of an infinite product would be NaN), so a masked key or a score of
// -infinity has weight 0; NaN stays NaN (a NaN-propagating maximum, one
// instruction).
__host__ __device__ __forceinline__ float exp_neg(float x) {
  constexpr float kHi = 1.44269502162933349609375f, kLo = 1.92596299112661746887e-8f, kLn2 = 0.693147180559945f;
  x = __builtin_elementwise_maximum(x, -128.0f);
  const float t = x * kHi;
  const float e = fmaf(x, kLo, fmaf(x, kHi, -t));
#ifdef __HIP_DEVICE_COMPILE__
  const float p = __builtin_amdgcn_exp2f(t);
#else
  const float p = exp2f(t);
#endif
  return fmaf(p * kLn2, e, p);
}
