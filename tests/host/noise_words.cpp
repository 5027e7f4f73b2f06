// Host run of NoiseGen::of_word (lowmachfhd_amd/csrc/stencils.h) at the ends of a word's range: the value
// is finite and its tail probability that of the word's uniform number.  Prints one line per failure;
// exit status 0 when there is none.  Built by tests/test_noise_host.py.
#include <cmath>
#include <cstdio>

#include "../../lowmachfhd_amd/csrc/stencils.h"

int main() {
  int bad = 0;
  const unsigned long long top = ~0ull >> 11;  // the largest m of (m + 1/2) 2^-53
  auto check = [&](unsigned long long m, double tail, bool upper) {
    // the probability of m, half an ulp of 1 to either side in the upper tail (the uniform number is a
    // double), and 1e-12 for the quantile's rounding (relative 1e-15, times x^2 = 70)
    const double x = lmfhd::NoiseGen::of_word(m << 11 | 0x7ffull);
    const double p = 0.5 * std::erfc((upper ? x : -x) * 0.70710678118654752440);
    const double slack = 1e-12 * tail + (upper ? std::ldexp(1.0, -54) * (1 + 1e-12) : 0.0);
    if (!(std::isfinite(x) && (upper ? x > 0 : x < 0) && std::fabs(p - tail) <= slack)) {
      ++bad;
      printf("m = %llu: %.17g, tail %.17g, expected %.17g\n", m, x, p, tail);
    }
  };
  for (unsigned long long k = 0; k < 4000; k = k < 64 ? k + 1 : k + k / 8) {
    const double tail = ((double)k + 0.5) * std::ldexp(1.0, -53);
    check(k, tail, false);
    check(top - k, tail, true);
  }
  printf("%d failures\n", bad);
  return bad != 0;
}
