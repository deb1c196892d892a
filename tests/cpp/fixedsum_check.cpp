// The deposit's fixed-point arithmetic (aprl_amd/csrc/fixedsum.hpp) on the
// host against 128-bit integers.
#define __host__
#define __device__
#define __forceinline__ inline
#include "fixedsum.hpp"

#include <cstdio>
#include <random>

using Wide = __int128;

static int failures = 0;
static void check(bool ok, const char* what) {
  if (!ok && ++failures <= 10) std::printf("failed: %s\n", what);
}

// m 2^e rounded to the nearest integer, ties to even
static Wide rounded(Wide m, int e) {
  if (e >= 0) return m << e;
  if (e <= -126) return 0;
  const Wide floor = m >> -e, rest = m - (floor << -e), half = Wide(1) << (-e - 1);
  return floor + (rest > half || (rest == half && (floor & 1)) ? 1 : 0);
}

static void checkProduct(double p, double w) {
  int ep, ew;
  const Wide mp = static_cast<Wide>(std::ldexp(std::frexp(p, &ep), 53));
  const Wide mw = static_cast<Wide>(std::ldexp(std::frexp(w, &ew), 53));
  const Wide exact = rounded(mp * mw, ep + ew - 106);
  check(static_cast<long long>(aprl_gpu::fixedPoint(p, w)) == static_cast<long long>(exact), "fixedPoint");
}

int main() {
  std::mt19937_64 rng(1);
  std::uniform_real_distribution<double> unit(-1.0, 1.0);
  for (int t = 0; t < 2000000; ++t) {
    const int scale = static_cast<int>(rng() % 63);  // |p| < 2^62
    checkProduct(std::ldexp(unit(rng), scale), unit(rng));
  }
  // products just below and above a half: 2^31 + 1/2 -+ 2^-k
  for (int k = 24; k < 50; ++k)
    for (int s = -1; s <= 1; s += 2)
      for (double n : {3.0, 5.0, 1025.0, 65537.0}) {
        const double w = 1.0 + s * std::ldexp(1.0, -k);
        for (double half : {0.5, 1.5, 2147483646.5, 2147483645.5}) checkProduct(half * n, w / n), checkProduct(half, w);
      }
  checkProduct(std::ldexp(1.0, 61), 1.0);
  checkProduct(-std::ldexp(1.0, 61), 1.0);
  checkProduct(0.0, 0.5);
  std::printf(failures ? "%d failures\n" : "fixed-point check passed\n", failures);
  return failures ? 1 : 0;
}
