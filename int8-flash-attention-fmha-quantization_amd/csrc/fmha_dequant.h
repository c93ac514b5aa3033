// De-quantisation of int8 values, shared by the quantisation kernels and the epilogues of the attention kernels.
#pragma once
#include <hip/hip_runtime.h>

#pragma clang fp contract(off)

namespace fmha_i8_gfx950 {

// inc/utils.hpp:53: (float)v / 127.0f * amax, in that order.  The quotient is formed without the division sequence: with
// 1/127 as the sum of two floats hi + lo, fma(v, hi, fl(v * lo)) rounds v (hi + lo) once, and for each of the 256 values
// of v that is the correctly rounded v / 127.0f (checked exhaustively by the tests).
__device__ __forceinline__ float dequant1(int v, float amax) {
  constexpr float kHi = 1.0f / 127.0f;
  constexpr float kLo = (float)(1.0 / 127.0 - (double)kHi);
  const float fv = (float)v;
  return __builtin_fmaf(fv, kHi, fv * kLo) * amax;
}
__device__ __forceinline__ unsigned cvt_pk_bf16(float a, float b) {  // to nearest even, NaN stays NaN
  unsigned r;
  asm("v_cvt_pk_bf16_f32 %0, %1, %2" : "=v"(r) : "v"(a), "v"(b));
  return r;
}

}  // namespace fmha_i8_gfx950
