// Device functions shared by the epilogues of the grouped GEMMs.
#pragma once

#include "moe_internal.h"

namespace moe {

// run.cpp:709-726: gate clamped from above, up clamped on both sides, then
// gate * sigmoid(alpha * gate) * (up + 1).  u1 is up + 1 already (the 1 rides
// with the bias).
__device__ __forceinline__ float swiglu_shifted(float g, float u1, float limit) {
  constexpr float kNegAlphaLog2e = -kAlpha * 1.4426950408889634f;
  g = fminf(g, limit);
  u1 = __builtin_amdgcn_fmed3f(u1, 1.0f - limit, 1.0f + limit);
  const float s = __builtin_amdgcn_rcpf(1.0f + __builtin_amdgcn_exp2f(kNegAlphaLog2e * g));
  return g * s * u1;
}

// two floats -> packed bf16, round to nearest even (v_cvt_pk_bf16_f32); a in the low half
__device__ __forceinline__ uint32_t pack_bf16(float a, float b) {
  typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
  typedef float f32x2 __attribute__((ext_vector_type(2)));
  f32x2 v = {a, b};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(v, bf16x2));
}

}  // namespace moe
