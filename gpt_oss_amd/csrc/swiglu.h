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

// A store of a GEMM's output.  PAST: past the caches, where the weights are read past them
// (gemm_streams_weights; bf16_stores_past has where not).  Written through L2 the output pushes out the rows that the tiles beside this one read,
// and its eviction gets in the way of the weights' stream.  us per GEMM (gate_up + down), plain stores / these:
// gemm_bf16.hip, 2880 x 2880, 896 tokens (672 active) at 32 experts 198 + 118 / 174 + 110, 6144 tokens at
// 128 experts 979 + 562 / 918 + 520 (the combine, which then reads from HBM, 66 / 72); gemm.hip, MXFP4, 800
// tokens at 128 experts 228 + 138 / 205 + 126, 256 at 32 experts 67 + 45 / 65 + 42.  Where the matrix cores are the time
// they gain nothing and the combine loses (4096 tokens at 32 experts 797 / 802 us per call), nor do
// they gain in gemm_fp4.hip (3000 tokens at 128 experts 615 / 620) and in stream.hip (64 tokens, MXFP4, 91 / 94).
template <bool PAST, typename V>
__device__ __forceinline__ void store_output(V *p, V v) {
  if constexpr (PAST) __builtin_nontemporal_store(v, p);
  else *p = v;
}

}  // namespace moe
