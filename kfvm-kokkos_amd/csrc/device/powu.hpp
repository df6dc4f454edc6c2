// x^y for 0 <= x <= 1 and y >= 0, the only range the HLLC shear factor
// (p_min/p_max)^M needs.  exp(y ln x) with
//   ln x : x = m 2^e, m in [1/sqrt 2, sqrt 2), ln m = 2 atanh(s) with
//          s = (m-1)/(m+1), |s| <= 0.1716, by its Taylor series to s^23
//          (truncation < 1e-18 relative);
//   exp t: Cody-Waite reduction t = n ln2 + r, |r| <= ln2/2, ln2 split in a
//          20-bit head (n*head exact) and a tail, exp r by Taylor to r^13
//          (truncation < 4e-18 relative), times 2^n.
// Error (against long-double powl, tests/test_powu.py): below 3.6e-15
// relative where x^y > 1e-3 (the rounding of t = y ln x carries over), and
// 1 - x^y, the quantity HLLC uses, within one ulp of 1 everywhere.
#pragma once

#ifdef __HIPCC__
#define KFVM_POWU_HD __host__ __device__
#else
#define KFVM_POWU_HD
#endif

#include <cmath>

namespace kfvm {

// exp(y (e ln 2 + 2 atanh s))
KFVM_POWU_HD inline double exp_y_ln(double s, int e, double y) {
  constexpr double LN2_HEAD = 0.6931467056274414;      // ln 2 with 32 trailing zero bits
  constexpr double LN2_TAIL = 4.7493250390316726e-07;  // ln 2 - LN2_HEAD
  constexpr double INV_LN2 = 1.4426950408889634;
  const double s2 = s * s;
  double p = 1.0 / 23.0;
  p = std::fma(p, s2, 1.0 / 21.0);
  p = std::fma(p, s2, 1.0 / 19.0);
  p = std::fma(p, s2, 1.0 / 17.0);
  p = std::fma(p, s2, 1.0 / 15.0);
  p = std::fma(p, s2, 1.0 / 13.0);
  p = std::fma(p, s2, 1.0 / 11.0);
  p = std::fma(p, s2, 1.0 / 9.0);
  p = std::fma(p, s2, 1.0 / 7.0);
  p = std::fma(p, s2, 1.0 / 5.0);
  p = std::fma(p, s2, 1.0 / 3.0);
  const double lnm = std::fma(2.0 * s * s2, p, 2.0 * s);
  const double de = double(e);
  const double t = y * (de * LN2_HEAD + (de * LN2_TAIL + lnm));
  if (t < -746.0) return 0.0;
  const double n = std::rint(t * INV_LN2);
  const double r = (t - n * LN2_HEAD) - n * LN2_TAIL;
  double q = 1.6059043836821613e-10;  // 1/13!
  q = std::fma(q, r, 2.08767569878681e-09);
  q = std::fma(q, r, 2.505210838544172e-08);
  q = std::fma(q, r, 2.755731922398589e-07);
  q = std::fma(q, r, 2.7557319223985893e-06);
  q = std::fma(q, r, 2.48015873015873e-05);
  q = std::fma(q, r, 0.0001984126984126984);
  q = std::fma(q, r, 0.001388888888888889);
  q = std::fma(q, r, 0.008333333333333333);
  q = std::fma(q, r, 0.041666666666666664);
  q = std::fma(q, r, 0.16666666666666666);
  q = std::fma(q, r, 0.5);
  q = std::fma(q, r, 1.0);
  q = std::fma(q, r, 1.0);
  return std::ldexp(q, int(n));
}

KFVM_POWU_HD inline double powu(double x, double y) {
  if (!(x > 0.0)) return x == 0.0 ? (y > 0.0 ? 0.0 : 1.0) : x;  // 0^y; NaN passes through
  int e;
  double m = std::frexp(x, &e);
  if (m < 0.70710678118654752) {
    m *= 2.0;
    e -= 1;
  }
  return exp_y_ln((m - 1.0) / (m + 1.0), e, y);
}

// (a/b)^y for 0 <= a <= b, b > 0 and y >= 0: as powu, with the ratio taken
// inside the logarithm, a = m 2^ea, b = n 2^eb, m/n brought into [1/sqrt 2,
// sqrt 2), s = (m-n)/(m+n): one division less than powu(a / b, y), and no
// rounding of the ratio (tests/test_pow_ratio.py: the bounds of powu).
#ifdef __HIPCC__
namespace dev {
__device__ inline double div_n(double a, double b);  // physics.hpp
__device__ inline double rcp_n(double x);
}
#endif

KFVM_POWU_HD inline double pow_ratio(double a, double b, double y) {
  if (!(a > 0.0)) return a == 0.0 ? (y > 0.0 ? 0.0 : 1.0) : a / b;  // 0^y; NaN passes through
  int ea, eb;
  double m = std::frexp(a, &ea);
  const double n = std::frexp(b, &eb);
  int e = ea - eb;
  if (m < 0.70710678118654752 * n) {
    m *= 2.0;
    e -= 1;
  } else if (m > 1.4142135623730951 * n) {
    m *= 0.5;
    e += 1;
  }
#ifdef __HIP_DEVICE_COMPILE__
  return exp_y_ln(dev::div_n(m - n, m + n), e, y);
#else
  return exp_y_ln((m - n) / (m + n), e, y);
#endif
}

// x^y for |y| <= 2^10 (an adiabatic exponent).  ln |x| as a head and a tail:
// |x| = m 2^e, m in [1/sqrt 2, sqrt 2), s = (m-1)/(m+1) with its remainder,
// 2 atanh(s) by Taylor to s^23; the product with y keeps its rounding error,
// which enters exp's reduced argument.  Within one ulp of powl
// (tests/test_pow_pos.py), the bound of the library's pow, of whose 190
// instructions it takes about 80.
KFVM_POWU_HD inline double pow_pos(double x, double y) {
  const double ax = std::fabs(x);
  constexpr double LN2_HEAD = 0.6931467056274414;
  constexpr double LN2_TAIL = 4.7493250390316726e-07;
  constexpr double INV_LN2 = 1.4426950408889634;
  int e;
  double m = std::frexp(ax, &e);
  if (m < 0.70710678118654752) {
    m *= 2.0;
    e -= 1;
  }
  const double f = m - 1.0, d = m + 1.0, dl = m - (d - 1.0);
#ifdef __HIP_DEVICE_COMPILE__
  const double r = dev::rcp_n(d);
#else
  const double r = 1.0 / d;
#endif
  const double s = f * r, sl = std::fma(-s, dl, std::fma(-s, d, f)) * r;
  const double z = s * s;
  double p = 1.0 / 23.0;
  p = std::fma(p, z, 1.0 / 21.0);
  p = std::fma(p, z, 1.0 / 19.0);
  p = std::fma(p, z, 1.0 / 17.0);
  p = std::fma(p, z, 1.0 / 15.0);
  p = std::fma(p, z, 1.0 / 13.0);
  p = std::fma(p, z, 1.0 / 11.0);
  p = std::fma(p, z, 1.0 / 9.0);
  p = std::fma(p, z, 1.0 / 7.0);
  p = std::fma(p, z, 1.0 / 5.0);
  p = std::fma(p, z, 1.0 / 3.0);
  // ln x = th + tl: e ln2_head (exact) + 2 s, then the small terms
  const double de = double(e), a = de * LN2_HEAD, b = 2.0 * s;
  const double sum = a + b, bb = sum - a;
  const double low = (a - (sum - bb)) + (b - bb) + std::fma(de, LN2_TAIL, 2.0 * std::fma(s * z, p, sl));
  const double th = sum + low, tl = low - (th - sum);
  const double t = y * th, u = std::fma(y, th, -t) + y * tl;
  const double n = std::rint(t * INV_LN2);
  const double w = std::fma(-n, LN2_HEAD, t) + (u - n * LN2_TAIL);
  double q = 1.6059043836821613e-10;  // 1/13!
  q = std::fma(q, w, 2.08767569878681e-09);
  q = std::fma(q, w, 2.505210838544172e-08);
  q = std::fma(q, w, 2.755731922398589e-07);
  q = std::fma(q, w, 2.7557319223985893e-06);
  q = std::fma(q, w, 2.48015873015873e-05);
  q = std::fma(q, w, 0.0001984126984126984);
  q = std::fma(q, w, 0.001388888888888889);
  q = std::fma(q, w, 0.008333333333333333);
  q = std::fma(q, w, 0.041666666666666664);
  q = std::fma(q, w, 0.16666666666666666);
  q = std::fma(q, w, 0.5);
  const double c = std::fma(q * w, w, w);  // e^w - 1
  double v = std::ldexp(1.0 + c, int(n));
  // zero, infinity, and a negative base (real for whole y only)
  const double inf = __builtin_inf();
  if (ax == 0.0 || ax == inf) v = y == 0.0 ? 1.0 : ((y > 0.0) == (ax == 0.0) ? 0.0 : inf);
  if (x < 0.0) {
    const double h = 0.5 * y;
    v = y != std::rint(y) ? __builtin_nan("") : (h != std::rint(h) ? -v : v);
  }
  return v;
}

}  // namespace kfvm
