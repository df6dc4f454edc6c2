// Host build of pow_pos (x^y) against long-double powl: the worst
// error in units of the last place of the result over densities and adiabatic
// exponents of both signs, and special values.
#include <cmath>
#include <cstdio>
#include <random>

#include "../kfvm-kokkos_amd/csrc/device/powu.hpp"

int main() {
  std::mt19937_64 g(5);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  double worst = 0.0;
  for (int i = 0; i < 4000000; i++) {
    const double x = i % 4 == 0 ? 0.05 + 3.0 * U(g) : (i % 4 == 1 ? std::exp(80.0 * (U(g) - 0.5))
                                                     : (i % 4 == 2 ? 1.0 + 1e-4 * (U(g) - 0.5) : 1.0 + 1e-12 * (U(g) - 0.5)));
    const double y = (i % 3 == 0 ? 1.4 : (i % 3 == 1 ? 5.0 / 3.0 : 1.0 + U(g))) * (i % 2 ? 1.0 : -1.0);
    const long double ref = powl((long double)x, (long double)y);
    const double v = kfvm::pow_pos(x, y);
    int e;
    std::frexp(double(ref), &e);
    worst = std::fmax(worst, double(fabsl((long double)v - ref)) / std::ldexp(1.0, e - 53));
  }
  const bool signs = kfvm::pow_pos(-2.0, 2.0) == 4.0 && kfvm::pow_pos(-2.0, 3.0) == -8.0 &&
                     kfvm::pow_pos(0.0, -1.4) == INFINITY && kfvm::pow_pos(INFINITY, -1.4) == 0.0 &&
                     kfvm::pow_pos(5e-324, 1.4) == 0.0 && kfvm::pow_pos(5e-324, 0.0) == 1.0;
  std::printf("%.6g %.17g %.17g %.17g %.17g %d %d %d\n", worst, kfvm::pow_pos(1.0, 1.4), kfvm::pow_pos(4.0, 0.5),
              kfvm::pow_pos(0.0, 1.4), kfvm::pow_pos(1e300, 3.0) == INFINITY ? 1.0 : 0.0,
              std::isnan(kfvm::pow_pos(-1.0, 1.4)) ? 1 : 0, std::isnan(kfvm::pow_pos(NAN, 1.4)) ? 1 : 0, signs ? 1 : 0);
  return 0;
}
