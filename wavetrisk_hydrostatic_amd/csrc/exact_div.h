// Division by a value whose reciprocal is at hand.
#pragma once
#include <hip/hip_runtime.h>

// a / d with r = 1 / d rounded to nearest: one remainder step makes the
// product the correctly rounded quotient (Markstein, IBM J. Res. Dev. 34,
// 1990) where nothing over- or underflows; an infinite a gives NaN.  Three
// operations instead of a division's eleven.
__device__ __forceinline__ double div_by(double a, double d, double r) {
  const double q = a * r;
  return __builtin_fma(__builtin_fma(-q, d, a), r, q);
}
