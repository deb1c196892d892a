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

}  // namespace aprl_gpu
