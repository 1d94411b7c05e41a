// Division by a divisor whose reciprocal is known: half the instructions of a
// division and half its latency, for divisors that several quotients share.
#pragma once
#include <hip/hip_runtime.h>

namespace fimhip {

// the reciprocal div_by takes: 1/s, or NaN (div_by then divides) where a
// remainder could leave the normal range
__device__ __forceinline__ double div_rcp(double s) { return s > 1.e-100 && s < 1.e100 ? 1. / s : __builtin_nan(""); }

// n / s for s > 0, from r = div_rcp(s), with the division's own rounding: two
// corrections of n r by its exact remainder (Markstein, IBM J. Res. Dev. 34,
// 1990: with r the double nearest to 1/s, a correction of a quotient that is
// within one unit in the last place ends on the nearest).  It divides where a
// remainder could underflow, and for inf and NaN.
__device__ __forceinline__ double div_by(double n, double s, double r) {
  double q = n * r;
  q = __builtin_fma(__builtin_fma(-q, s, n), r, q);
  q = __builtin_fma(__builtin_fma(-q, s, n), r, q);
  if (!(fabs(q) < 1.e250 && fabs(n) > 1.e-180)) {
    if (n == 0.) q = n;
    else q = n / s;
  }
  return q;
}

}  // namespace fimhip
