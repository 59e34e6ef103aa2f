// gelu on the store of a product.
#pragma once
#include "castle_tiles.h"

namespace castle {

// Phi(x) = erfc(-x / sqrt 2) / 2.  For 16-bit outputs from the Chebyshev fit of Numerical Recipes (erfcc, fractional error
// below 1.2e-7 everywhere); the library's erff takes three times the instructions, which a store of 16384 x 2048 felt
// with 8 us.
template <typename T> __device__ __forceinline__ float normal_cdf(float x) {
  if constexpr (sizeof(T) == 4) {
    return 0.5f * (1.f + erff(x * 0.70710678f));
  } else {
    const float z = fabsf(x) * 0.70710678f, t = fast_rcp(__builtin_fmaf(0.5f, z, 1.f));
    float p = 0.17087277f;
    p = __builtin_fmaf(p, t, -0.82215223f);
    p = __builtin_fmaf(p, t, 1.48851587f);
    p = __builtin_fmaf(p, t, -1.13520398f);
    p = __builtin_fmaf(p, t, 0.27886807f);
    p = __builtin_fmaf(p, t, -0.18628806f);
    p = __builtin_fmaf(p, t, 0.09678418f);
    p = __builtin_fmaf(p, t, 0.37409196f);
    p = __builtin_fmaf(p, t, 1.00002368f);
    p = __builtin_fmaf(p, t, -1.26551223f);
    const float e = 0.5f * t * fast_exp2(kLog2e * (p - z * z));
    return x < 0.f ? e : 1.f - e;
  }
}
template <typename T> __device__ __forceinline__ float gelu(float x) { return x * normal_cdf<T>(x); }
template <typename T> __device__ __forceinline__ float gelu_slope(float x) {
  return normal_cdf<T>(x) + x * 0.3989422804f * fast_exp2(-0.5f * kLog2e * x * x);
}

}  // namespace castle
