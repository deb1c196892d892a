// Fixed-point arithmetic of the deposit's current sums (host and device).
#pragma once

#include <cmath>

namespace aprl_gpu {

// part1 * w rounded to an integer, |part1 * w| < 2^62: the sum with 1.5 2^84
// leaves the nearest multiple m of 2^32 in its low word, and that with
// 1.5 2^52 - m (exact: a multiple of 2^32 below 2^63) the rest, the product
// rounded once (an llrint of the rounded product takes twice the
// instructions, and its product a rounding of its own).
__host__ __device__ __forceinline__ unsigned long long fixedPoint(double part1, double w) {
#pragma clang fp contract(off)
  const double hi = std::fma(part1, w, 0x1.8p84);
  const double lo = std::fma(part1, w, (0x1.8p84 - hi) + 0x1.8p52);
  const unsigned long long h = __builtin_bit_cast(unsigned long long, hi);
  const unsigned long long l = __builtin_bit_cast(unsigned long long, lo);
  return ((h << 32) + l) - 0x4338000000000000ull;
}

// The quintic's compensation (quinticCompensation): numerators over
// 1024 27 7, the weights' common denominator.
constexpr double kQuinticDen = 193536.;
constexpr double kQuinticNum[7] = {-1571., 17322., -95469., 352972., -95469., 17322., -1571.};

// (a 2^32 + b) / kQuinticDen rounded to the nearest integer (halves up), for
// whole a, b: the sums of kQuinticNum times the high words (|.| <= 2^30) and
// the low words (< 2^32) of raw sums, exact in FP64 (the numerators' absolute
// values add up to 581696 < 2^19.2). The high sum's quotient leaves a
// remainder of at most half the denominator, which joins the low sum below
// 2^52; that sum's quotient is off the nearest integer only where it halves.
__host__ __device__ __forceinline__ long long quinticQuotient(double a, double b) {
#pragma clang fp contract(off)
  constexpr double inverse = 1.0 / kQuinticDen;
  const double high = std::fma(a, inverse, 0x1.8p52);
  const double left = std::fma(std::fma(-kQuinticDen, high - 0x1.8p52, a), 0x1p32, b);
  const double low = std::fma(left, inverse, 0x1.8p52);
  const double rest = std::fma(-kQuinticDen, low - 0x1.8p52, left);
  const unsigned long long h = __builtin_bit_cast(unsigned long long, high);
  const unsigned long long l = __builtin_bit_cast(unsigned long long, low);
  return static_cast<long long>(((h << 32) + l) - 0x4338000000000000ull + (2.0 * rest >= kQuinticDen ? 1 : 0));
}

}  // namespace aprl_gpu
