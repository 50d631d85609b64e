// div_rn.h — x / s correctly rounded in fp32 from the correctly rounded reciprocal of s.
//
// Markstein's quotient: with rs = RN(1 / s), q = RN(x rs) is within one ulp of x / s, the
// residual r = x - s q is exact when computed by one fma, and RN(q + r rs) = RN(x / s).  The
// conditions are that the residual neither underflows nor overflows — here x and q both in
// [2^-100, 2^100] — and a quotient of two fp32 values is never a rounding midpoint.  Outside
// that range (zero, tiny or huge operands, NaN, inf, a zero or denormal scale) the division
// itself is taken.  Three operations instead of the dozen of an IEEE division, for kernels
// that divide every element by one scale.
#pragma once

#include <hip/hip_runtime.h>

namespace rxmet {

__device__ __forceinline__ float div_rn(float x, float s, float rs) {
  const float q = x * rs;
  const float ax = fabsf(x), aq = fabsf(q);
  if (ax >= 0x1p-100f && ax <= 0x1p100f && aq >= 0x1p-100f && aq <= 0x1p100f)
    return fmaf(fmaf(-q, s, x), rs, q);
  return x / s;
}

// The quotients of a vector of E elements with one check for all of them: with 1 / s in
// [2^-60, 2^60] and every x zero or in [2^-40, 2^40], x and q are in div_rn's range; the residual
// steps lose the sign of a zero only, which q has.  Else the elements are divided one by one.
// (div_rn per element spends ten instructions and a branch on its four comparisons, and its branch
// takes the zeros of a rectified activation through the division.)
template <int E>
__device__ __forceinline__ void div_rn_vec(const float (&x)[E], float s, float rs, float (&t)[E]) {
  unsigned lo = ~0u, hi = 0u;  // of |x| as integers (NaN is the largest), zero wrapped past lo
#pragma unroll
  for (int k = 0; k < E; ++k) {
    const float q = x[k] * rs;
    t[k] = copysignf(fmaf(fmaf(-q, s, x[k]), rs, q), q);
    const unsigned u = __builtin_bit_cast(unsigned, x[k]) & 0x7fffffffu;
    lo = min(lo, u - 1u);
    hi = max(hi, u);
  }
  const float ar = fabsf(rs);
  const bool in = ar >= 0x1p-60f && ar <= 0x1p60f &&
                  lo >= __builtin_bit_cast(unsigned, 0x1p-40f) - 1u &&
                  hi <= __builtin_bit_cast(unsigned, 0x1p40f);
  if (!in) {
#pragma unroll
    for (int k = 0; k < E; ++k) t[k] = div_rn(x[k], s, rs);
  }
}

}  // namespace rxmet
