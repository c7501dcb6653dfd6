// Correctly rounded float quotients by a divisor whose reciprocal is known,
// for the exact traversal's slab test: a ray divides by the same three
// direction components at every node. No HIP types, so the CPU check
// (tests/cpu/exact_div_check.cpp) runs this very code.
#ifndef MUONX_DEVICE_EXACT_DIV_H_
#define MUONX_DEVICE_EXACT_DIV_H_

#include <cmath>

#if defined(__HIPCC__) || defined(__HIP__)
#define MX_DIV_HD __host__ __device__ __forceinline__
#else
#define MX_DIV_HD inline
#endif

namespace muonx {

// a / d rounded to nearest, given inv = 1 / d rounded to nearest: the
// product a * inv (within two ulps of the quotient) corrected once by its
// exact remainder (P. Markstein, "Computation of elementary functions on the
// IBM RISC System/6000 processor", 1990). The sum before the last rounding
// is within 2^-23 ulp of the quotient, so it rounds as the quotient does
// unless that lies within 2^-23 ulp of a midpoint; the CPU check enumerates
// every pair of significands that does. Needs a remainder, a reciprocal and a
// quotient that neither overflow nor lose bits to underflow: DivisorOk for d,
// and a zero or 2^-99 <= |a| <= 2^61.
// Three operations (7 issue cycles on gfx950) against the eleven (about 50
// cycles) of an IEEE division.
MX_DIV_HD float QuotientByReciprocal(float a, float d, float inv) {
  const float q = a * inv;
  return __builtin_fmaf(__builtin_fmaf(-q, d, a), inv, q);
}

// Divisors of QuotientByReciprocal: a zero one gives NaN, which the slab
// test ignores (the axis is skipped, as in muon/bounds.cc:98-100).
MX_DIV_HD bool DivisorOk(float d) {
  const float m = __builtin_fabsf(d);
  return m == 0.0f || (m >= 0x1p-60f && m <= 0x1p20f);
}

// Coordinates whose differences are dividends of QuotientByReciprocal: the
// difference of two such floats is zero, or a multiple of 2^-99 of at most
// 2^61.
MX_DIV_HD bool CoordinateOk(float x) {
  const float m = __builtin_fabsf(x);
  return m == 0.0f || (m >= 0x1p-76f && m <= 0x1p60f);
}

}  // namespace muonx

#endif
