// Host build of pow_ratio ((a/b)^y, 0 <= a <= b, y >= 0) against long-double
// powl: the quantities powu_check.cpp prints.
#include <cmath>
#include <cstdio>
#include <random>

#include "../kfvm-kokkos_amd/csrc/device/powu.hpp"

int main() {
  std::mt19937_64 g(11);
  std::uniform_real_distribution<double> U(0.0, 1.0);
  double worstRel = 0.0, worstAbs = 0.0;
  for (int i = 0; i < 3000000; i++) {
    const double b = std::exp(60.0 * (U(g) - 0.5));
    const double a = b * (i % 3 == 0 ? U(g) : (i % 3 == 1 ? std::exp(-40.0 * U(g)) : 1.0 - 1e-6 * U(g)));
    const double y = i % 2 ? 60.0 * U(g) : 3.0 * U(g);
    const long double ref = powl((long double)a / (long double)b, (long double)y);
    const double x = kfvm::pow_ratio(a, b, y);
    if (ref > 1e-3L) worstRel = std::fmax(worstRel, double(fabsl((x - ref) / ref)) / 1.1102230246251565e-16);
    worstAbs = std::fmax(worstAbs, std::fabs(double((1.0L - (long double)x) - (1.0L - ref))));
  }
  std::printf("%.6g %.6g %.17g %.17g %.17g %.17g %.17g\n", worstRel, worstAbs, kfvm::pow_ratio(2.5, 2.5, 3.5),
              kfvm::pow_ratio(0.3, 0.7, 0.0), kfvm::pow_ratio(0.0, 3.0, 2.0), kfvm::pow_ratio(0.75, 3.0, 0.5),
              kfvm::pow_ratio(1e-300, 1e300, 3.0));
  return 0;
}
