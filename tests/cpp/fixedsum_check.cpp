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

// A column of raw sums (below 2^62 over the weights' bound 3.125, the tile's
// scale) under the quintic's weights, rounded to the nearest integer.
static void checkColumn(const long long raw[7]) {
  double a = 0.0, b = 0.0;
  const Wide den = static_cast<Wide>(aprl_gpu::kQuinticDen);
  Wide t = den / 2;
  for (int q = 0; q < 7; ++q) {
    a = std::fma(aprl_gpu::kQuinticNum[q], static_cast<double>(static_cast<int>(raw[q] >> 32)), a);
    b = std::fma(aprl_gpu::kQuinticNum[q], static_cast<double>(static_cast<unsigned>(raw[q])), b);
    t += static_cast<Wide>(aprl_gpu::kQuinticNum[q]) * raw[q];
  }
  Wide nearest = t / den;
  if (t < 0 && nearest * den != t) --nearest;
  check(static_cast<Wide>(aprl_gpu::quinticQuotient(a, b)) == nearest, "quotient");
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
  // the weights: numerators over the denominator against the moments' formula
  const double p5 = 5., wa = p5 / 6., wb = 3 * p5 / 40. + p5 * (p5 - 1) / 72.,
               wd = 5 * p5 / 112. + p5 * (p5 - 1) / 80. + p5 * (p5 - 1) * (p5 - 2) / 1296.;
  const double weight[7] = {-wd / 64., wb / 16. + 3 * wd / 32., -wa / 4. - wb / 4. - 15 * wd / 64.,
                            1 + wa / 2. + 3 * wb / 8. + 5 * wd / 16., -wa / 4. - wb / 4. - 15 * wd / 64.,
                            wb / 16. + 3 * wd / 32., -wd / 64.};
  for (int q = 0; q < 7; ++q)
    check(std::fabs(aprl_gpu::kQuinticNum[q] / aprl_gpu::kQuinticDen - weight[q]) < 1e-15, "weights");
  const long long top = static_cast<long long>(0x1p62 / 3.125);
  for (int t = 0; t < 2000000; ++t) {
    long long raw[7];
    const int bits = static_cast<int>(rng() % 60);
    for (long long& r : raw) r = (static_cast<long long>(rng()) % top) >> bits;
    checkColumn(raw);
  }
  const long long ends[3][7] = {{-top, top, -top, top, -top, top, -top}, {top, -top, top, -top, top, -top, top},
                                {0, 0, 0, 0, 0, 0, 0}};
  for (const auto& raw : ends) checkColumn(raw);
  for (long long n = -400000; n <= 400000; ++n) {  // every remainder
    const long long raw[7] = {n, 0, 0, 0, 0, 0, 0};
    checkColumn(raw);
  }
  std::printf(failures ? "%d failures\n" : "fixed-point check passed\n", failures);
  return failures ? 1 : 0;
}
