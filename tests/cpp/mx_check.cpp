// Host checks of the matrix-core rejection's rules (csrc/mx_rules.hpp).
// Returns 0, or names the first case that fails.
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <limits>
#include <random>

#include "mx_rules.hpp"

using namespace gcr;

// Every operand is a number of magnitude at most 1 whatever the model holds:
// the test's answer is the sign of a multiply-add, so a NaN would be one.
template <int KIND>
static long check_normalise(std::mt19937_64& rng) {
  const double inf = std::numeric_limits<double>::infinity(), nan = std::numeric_limits<double>::quiet_NaN();
  const double odd[] = {inf, -inf, nan, -nan, 1e306, -1.7e308, 5e-324, 1e-310, -1e-301, 0.0, 1e300, 1e-300};
  std::uniform_real_distribution<double> u(-1.0, 1.0);
  long zero = 0;
  for (int trial = 0; trial < 200000; ++trial) {
    double M[9], F[9];
    const double size = std::pow(10.0, 6.0 * u(rng));
    for (double& v : M) v = size * u(rng);
    const int odds = (int)(rng() % 4);  // up to three odd entries, or all
    for (int k = 0; k < odds; ++k) M[rng() % 9] = odd[rng() % 12];
    if (trial % 16 == 0)
      for (double& v : M) v = odd[rng() % 12];
    const double s = std::ldexp(1.0, (int)(rng() % 40) - 20);
    const bool test = trial % 8 != 0;
    mx_normalise<KIND>(M, s, test, F);
    bool finite = true;
    double mx = 0.0;
    for (int k = 0; k < 9; ++k) {
      finite = finite && std::isfinite(M[k]);
      mx = std::fmax(mx, std::fabs(F[k]));
      if (!(std::fabs(F[k]) <= 1.0 + 1e-15)) {
        std::printf("FAIL kind %d trial %d: entry %d is %g (model entry %g)\n", KIND, trial, k, F[k], M[k]);
        std::exit(1);
      }
    }
    if ((!finite || !test) && mx != 0.0) {
      std::printf("FAIL kind %d trial %d: operands of a model that is not tested\n", KIND, trial);
      std::exit(1);
    }
    if (mx == 0.0) ++zero;
    else if (mx < 1.0 - 1e-15) {
      std::printf("FAIL kind %d trial %d: largest entry %g\n", KIND, trial, mx);
      std::exit(1);
    }
  }
  return zero;
}

int main() {
  std::mt19937_64 rng(7);
  const long z1 = check_normalise<1>(rng), z0 = check_normalise<0>(rng);
  std::printf("ok, untested %ld %ld\n", z1, z0);
  return z1 > 1000 && z0 > 1000 && z1 < 190000 ? 0 : 1;
}
