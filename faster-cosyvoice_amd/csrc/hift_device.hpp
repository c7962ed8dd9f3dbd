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

}  // namespace
}  // namespace fcv
