// Many quotients of one divisor; plain functions, so that a CPU program can call them.
#pragma once

#include <math.h>

#if !defined(__HIPCC__)
#define __host__
#define __device__
#define __forceinline__ inline
#endif

namespace marian_hip {

// a / s from r = 1.0f / s, s positive: three operations where a division takes eleven.  The residual correction with a correctly rounded
// reciprocal gives the correctly rounded quotient (P. Markstein, "Computation of elementary functions on the IBM RISC
// System/6000 processor", 1990), so the bits are the division's (tests/test_shared_quotient.py, for odd divisors, and
// tests/test_shared_quotient_even.py: every pair of significands whose quotient lies close to a rounding edge).  The callers keep to magnitudes in which no step under- or overflows.  A zero keeps its
// sign: what is added to it is the remainder, which is +0, times -r (tests/test_quotients_of_zero.py).
constexpr float kQuotientLeast = 0x1p-60f, kQuotientMost = 0x1p60f;  // magnitudes of dividends that are not zero
constexpr float kDivisorLeast = 0x1p-40f, kDivisorMost = 0x1p40f;
__host__ __device__ __forceinline__ float shared_quotient(float a, float s, float r) {
  const float q = a * r;
  return fmaf(fmaf(q, s, -a), -r, q);
}
// The least of several of these is at least kDividendLeast where all dividends but the zeros have a magnitude of at least kQuotientLeast.
__host__ __device__ __forceinline__ unsigned dividend_order(float a) { return (__builtin_bit_cast(unsigned, a) & 0x7FFFFFFFu) - 1u; }
constexpr unsigned kDividendLeast = ((127u - 60u) << 23) - 1u;

}  // namespace marian_hip
