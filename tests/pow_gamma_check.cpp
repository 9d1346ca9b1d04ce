// Host check of pow_gamma (pyminiweather_amd/csrc/pmw_pow.h) against a
// 113-bit reference (quadmath powq, rounded once to double).
// Usage: pow_gamma_check N lo hi -> prints "N not_correctly_rounded special_mismatches
// max_relative_error_of_pow_gamma_minus_one"
#include <quadmath.h>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include "pmw_pow.h"
static const double kGam = 1.40027894002789400278940027894;
static bool same(double a, double b) { return (std::isnan(a) && std::isnan(b)) || a == b; }
int main(int argc, char** argv) {
  if (argc < 4) return 2;
  const long long n = atoll(argv[1]);
  const double lo = atof(argv[2]), hi = atof(argv[3]);
  uint64_t s = 0x9E3779B97F4A7C15ULL;
  long long bad = 0;
  double m1 = 0.0;
  for (long long i = 0; i < n; ++i) {
    s ^= s << 13; s ^= s >> 7; s ^= s << 17;
    const double u = (double)(s >> 11) * 0x1p-53;
    const double x = exp(log(lo) + u * (log(hi) - log(lo)));
    bad += pmw::pow_gamma(x) != (double)powq((__float128)x, (__float128)kGam);
    const __float128 ex = powq((__float128)x, (__float128)(kGam - 1.0));
    m1 = fmax(m1, fabs((double)(((__float128)pmw::pow_gamma_minus_one(x) - ex) / ex)));
  }
  int special = 0;
  // signs, zeros, infinities, NaN, subnormals, the edges of overflow, and the
  // first and last argument of table intervals and binades
  const double xs[] = {0.0, -0.0, -1.0, -300.0, INFINITY, -INFINITY, NAN, -NAN, 5e-324, 1e-310,
                       0x1p731, 0x1.2p731, 0x1.3p731, 0x1p732, 1e300, 1e308, -1e308, -1e-310};
  for (double x : xs) {
    const double a = pmw::pow_gamma(x);
    const double b = x < 0.0 && !std::isinf(x) ? NAN : (double)powq((__float128)x, (__float128)kGam);
    special += !same(a, b);
    const double c = pmw::pow_gamma_minus_one(x);  // NaN unless positive and normal
    special += std::isnan(c) == (x >= 0x1p-1022 && std::isfinite(x));
  }
  for (int e = -600; e <= 700; e += 25)
    for (int j = 0; j < 512; ++j)
      for (int d = -1; d <= 1; ++d) {
        double x = ldexp(1.0 + j / 512.0, e);
        x = d < 0 ? nextafter(x, 0.0) : d > 0 ? nextafter(x, INFINITY) : x;
        bad += pmw::pow_gamma(x) != (double)powq((__float128)x, (__float128)kGam);
      }
  printf("%lld %lld %d %.6g\n", n, bad, special, m1);
  return 0;
}
