// Host check of the range of pow_gamma's table (pyminiweather_amd/csrc/pmw_pow.h).
// Usage: pow_table_check X... -> prints "arguments_outside not_correctly_rounded
// edges": of the arguments X how many the table alone does not serve, and of the
// first and last arguments of every interval of its binades and the two beyond
// (edges of them) how many powers differ from the rounded 113-bit one.
#include <quadmath.h>
#include <cmath>
#include <cstdio>
#include <cstdlib>
#include "pmw_pow.h"
int main(int argc, char** argv) {
  constexpr unsigned entries = sizeof(pmw::powt::kGamQ) / sizeof(pmw::powt::kGamQ[0]);
  int outside = 0, bad = 0, edges = 0;
  for (int i = 1; i < argc; ++i) {
    double s, l;
    unsigned k;
    pmw::pow_gamma_entry(atof(argv[i]), s, l, k);
    outside += k >= entries;
  }
  for (int e = -8; e <= 11; ++e)
    for (int j = 0; j < 512; ++j)
      for (int last = 0; last < 2; ++last) {
        double x = ldexp(1.0 + (j + last) / 512.0, e);
        if (last) x = nextafter(x, 0.0);
        ++edges;
        bad += pmw::pow_gamma(x) !=
               (double)powq((__float128)x, (__float128)1.40027894002789400278940027894);
      }
  printf("%d %d %d\n", outside, bad, edges);
  return 0;
}
