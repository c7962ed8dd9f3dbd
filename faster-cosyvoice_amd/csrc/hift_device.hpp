// Device helpers shared by the HiFT vocoder kernels (hift.hip, hift_split.hip).
#pragma once

#include "hift.hpp"

namespace fcv {
namespace {

// largest d with cu[d] <= row
__device__ __forceinline__ int doc_of(const int32_t* cu, int n_docs, int row) {
  int lo = 0, hi = n_docs - 1;
  while (lo < hi) {
    const int mid = (lo + hi + 1) >> 1;
    if (cu[mid] <= row) lo = mid; else hi = mid - 1;
  }
  return lo;
}

// Snake(x) = x + sin(a x)^2 / (a + 1e-9), with inv = 1 / (a + 1e-9) precomputed in fp32.
// sin by v_sin_f32 on the fractional part of the argument in turns (v_fract_f32 is exact).
__device__ __forceinline__ float snake(float x, float a, float inv) {
  const float turns = (x * a) * 0.15915494309189535f;
  const float s = __builtin_amdgcn_sinf(__builtin_amdgcn_fractf(turns));
  return fmaf(inv, s * s, x);
}

// |v|, or 0 where v is infinite or NaN: a tensor's scale is that of its finite values
__device__ __forceinline__ float finite_abs(float v) {
  const float a = fabsf(v);
  return a <= 3.402823466e38f ? a : 0.0f;
}

// A tensor's largest finite magnitude per document is kept as the maximum of kAmaxSub values (fp32
// bits, which order like integers), kAmaxStride words apart: the workgroups of a launch raise
// different ones, since atomics on one address run one after the other (some 25 ns each: a
// Snake pass over 8 k rows took 53 us against 5 with one value).
__device__ __forceinline__ uint32_t* amax_word(uint32_t* amax, int doc, int sub) {
  return amax + ((long)doc * kAmaxSub + (sub & (kAmaxSub - 1))) * kAmaxStride;
}
__device__ __forceinline__ void raise_amax(uint32_t* amax, int doc, int sub, float v) {
  if (v > 0.0f) atomicMax(amax_word(amax, doc, sub), __float_as_uint(v));
}
// the maximum over the wave, valid in every lane
__device__ __forceinline__ float wave_max(float v) {
  v = fmaxf(v, dpp_f<0xB1>(v));
  v = fmaxf(v, dpp_f<0x4E>(v));
  v = fmaxf(v, dpp_f<0x141>(v));
  v = fmaxf(v, dpp_f<0x140>(v));
  const auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  v = fmaxf(__uint_as_float(r[0]), __uint_as_float(r[1]));
  const auto q = __builtin_amdgcn_permlane32_swap(__float_as_uint(v), __float_as_uint(v), false,
                                                  false);
  return fmaxf(__uint_as_float(q[0]), __uint_as_float(q[1]));
}

}  // namespace
}  // namespace fcv
