// Correctly rounded 1 / b and a / b in few instructions, for b well inside the
// normal range (the geometry of the 2-D patches: four quotients of a point
// share one reciprocal, 25 instructions instead of four full divisions' 44).
//
// Markstein's theorems (IBM J. Res. Dev. 34, 1990): a residual step from a
// reciprocal within one ulp rounds correctly unless the significand of b is all
// ones, and with y the rounded reciprocal a residual step from a faithful
// quotient rounds correctly; the first of the two steps makes it faithful.  For
// the all-ones significand the reciprocal is right if its seed is.  v_rcp_f32 of
// gfx950 gives that seed rounded correctly: over all 2^23 significands at five
// exponents, 897,675 of its results are one ulp off and none more, and the
// refined reciprocals and 64 quotients of each all equal the IEEE division's.
// A quotient of -0 is +0.
#pragma once

#include <hip/hip_runtime.h>

namespace sfx {

// y: 1 / b within one ulp
__device__ __forceinline__ float refined_reciprocal(float b, float y) {
  y = fmaf(fmaf(-b, y, 1.0f), y, y);
  return fmaf(fmaf(-b, y, 1.0f), y, y);
}
__device__ __forceinline__ float reciprocal(float b) { return refined_reciprocal(b, __builtin_amdgcn_rcpf(b)); }
// y: reciprocal(b)
__device__ __forceinline__ float quotient(float a, float b, float y) {
  float q = a * y;
  q = fmaf(fmaf(-b, q, a), y, q);
  return fmaf(fmaf(-b, q, a), y, q);
}

}  // namespace sfx
