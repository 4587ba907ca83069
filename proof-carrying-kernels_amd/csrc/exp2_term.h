// 2^(hi + lo) in FP32 for the set checker's softmax terms, gfx950 device code.
//
// The argument is an unevaluated sum, |lo| at most a few ulps of hi, hi <= 0.  It is reduced to
// k = rint(hi) and f = (hi - k) + lo, |f| <= 1/2 + 2^-16 (hi - k is exact), so lo needs no second
// product after the exponential, and 2^f = 1 + f P(f) with P of degree 5: a least-squares fit of
// 2^f on [-1/2, 1/2] iterated towards the smallest largest relative error, its coefficients
// rounded to FP32 from the lowest up with the others fitted again after each.  The polynomial is
// within 2^-28.3 and its mean error over f is 6e-13; the result is within 0.95 ulp (0.90 measured),
// rounded to nearest in the last step (no systematic part), exactly 1 at 0, and subnormal results
// are kept down to 2^-149.
//
// Against the exponential unit's v_exp_f32 with lo applied afterwards, which takes about as many
// issue slots (a quarter-rate instruction and two more for lo; check_topp_gpu of 64 x 151,936 logits
// within 2%): that truncates in part, which left the top-p masses a mean signed error of 4.0e-10 at
// T = 1 against expf's 1.4e-10 and 2e-13 here, and it gives 0 below 2^-126.

#pragma once

#include <hip/hip_runtime.h>

namespace pck {

__device__ __forceinline__ float exp2_pair(float hi, float lo) {
  const float k = __builtin_rintf(hi);
  const float f = (hi - k) + lo;
  float p = 0x1.416b52p-13f;
  p = __builtin_fmaf(p, f, 0x1.5f082ep-10f);
  p = __builtin_fmaf(p, f, 0x1.3b2de0p-7f);
  p = __builtin_fmaf(p, f, 0x1.c6af7cp-5f);
  p = __builtin_fmaf(p, f, 0x1.ebfbdcp-3f);
  p = __builtin_fmaf(p, f, 0x1.62e430p-1f);
  const float r = __builtin_ldexpf(__builtin_fmaf(p, f, 1.0f), static_cast<int>(k));
  // below half the smallest subnormal (and where hi is -inf, or NaN from an infinite difference): 0
  return hi >= -150.0f ? r : 0.0f;
}

}  // namespace pck
