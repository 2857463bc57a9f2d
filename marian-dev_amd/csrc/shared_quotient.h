// Many quotients of one divisor; plain functions, so that a CPU program can call them.
#pragma once

#include <math.h>

#if !defined(__HIPCC__)
#define __host__
#define __device__
#define __forceinline__ inline
#endif

namespace marian_hip {

// a / s from r = 1.0f / s: three operations where a division takes eleven.  The residual correction with a correctly rounded
// reciprocal gives the correctly rounded quotient (P. Markstein, "Computation of elementary functions on the IBM RISC
// System/6000 processor", 1990), so the bits are the division's (tests/test_shared_quotient.py: every pair of significands whose
// quotient lies close to a rounding edge).  The callers keep to magnitudes in which no step under- or overflows; a quotient
// of zero comes out as +0 whatever the signs, so they take the division where that could differ.
constexpr float kQuotientLeast = 0x1p-60f, kQuotientMost = 0x1p60f;  // magnitudes of dividends that are not zero
constexpr float kDivisorLeast = 0x1p-40f, kDivisorMost = 0x1p40f;
__host__ __device__ __forceinline__ float shared_quotient(float a, float s, float r) {
  const float q = a * r;
  return fmaf(fmaf(-q, s, a), r, q);
}

}  // namespace marian_hip
