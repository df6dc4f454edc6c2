// Mirror-symmetric form of the WENO weights: parity.hpp's slots for the full
// and centre substencils, and for the biased ones, which are symmetric in the
// two axes across their bias only and are each other's mirror image along it.
//
// With T the butterfly over all axes, the values of the biased substencil on
// the negative side of axis b, transformed across b only, are (sum - difference)
// / 2 of the slot pairs of axis b, those on the positive side (sum + difference)
// / 2 (the factor is folded into the coefficients), so no second copy of the
// stencil is kept.  One coefficient list serves both sides.
//   derivative rows   a derivative's row is nonzero in one parity class only
//                     (two for a pure second derivative of the full and centre
//                     substencils, whose weights mix them)
//   points            the even and odd part along b of the negative side's
//                     weights at the two points +-x_b; the positive side's odd
//                     part has the other sign
// 3D: 142 + 3 x 2 x 64 products for the smoothness indicators instead of 19 x
// 106, and 40 + 3 x 44 per 8 points instead of 8 x 106.
#pragma once

#include <algorithm>
#include <cmath>
#include <vector>

#include "parity.hpp"

namespace kfvm {

template <int D>
struct DerivRows {
  int ex[SInfo<D>::I][3];  // exponents of the derivative of each row
};
template <int D>
constexpr DerivRows<D> make_deriv_rows() {
  DerivRows<D> r{};
  int n = 0;
  for (int t = 1; t <= SInfo<D>::nDeriv; t++)
    for (int i = 0; i <= t; i++)
      for (int j = (D == 2 ? t - i : 0); j <= t - i; j++) {
        r.ex[n][0] = i;
        r.ex[n][1] = j;
        r.ex[n][2] = t - i - j;
        n++;
      }
  return r;
}

// Positions of the coefficients in the list (-1: no product).
template <int D>
struct WenoParityDeriv {
  int row[2][SInfo<D>::I][SInfo<D>::C];   // full and centre substencil: by slot
  int bia[D][SInfo<D>::I][SInfo<D>::Cb];  // axis b: by cell of the negative side
  int count;
};
template <int D>
constexpr WenoParityDeriv<D> make_weno_parity_deriv() {
  using S = SInfo<D>;
  constexpr auto st = make_stencil_tables<D>();
  constexpr auto pt = make_parity_tables<D>();
  constexpr auto dr = make_deriv_rows<D>();
  WenoParityDeriv<D> w{};
  int k = 0;
  for (int s = 0; s < 2; s++)
    for (int i = 0; i < S::I; i++) {
      int p = 0, deg = 0, second = -1;
      for (int d = 0; d < D; d++) {
        p |= (dr.ex[i][d] & 1) << d;
        deg += dr.ex[i][d];
        if (dr.ex[i][d] == 2) second = d;
      }
      for (int n = 0; n < S::C; n++) {
        const bool in = s == 0 || n < S::Cc;
        const bool on = pt.neg[n] == p || (deg == 2 && second >= 0 && pt.neg[n] == 1 << second);
        w.row[s][i][n] = in && on ? k++ : -1;
      }
    }
  for (int b = 0; b < D; b++)
    for (int i = 0; i < S::I; i++)
      for (int m = 0; m < S::Cb; m++) {
        bool on = true;
        for (int r = 1; r < D; r++)  // the rows are those of the x-biased substencil, its axes permuted
          if (((pt.neg[st.sub[2 * b][m]] >> parity_frame_axis(b, r)) & 1) != (dr.ex[i][r] & 1)) on = false;
        w.bia[b][i][m] = on ? k++ : -1;
      }
  w.count = k;
  return w;
}

// The same for the points of face axis A, or the interior points (A = -1),
// counted from the group's first coefficient.  bia: even part; the odd part,
// if the points are not zero along b, follows it.
template <int D, int NQ, int A>
struct WenoParityPoints {
  static constexpr int TYPES = A >= 0 ? parity_face_types(D, NQ) : parity_cell_types(D, NQ);
  int row[2][TYPES][SInfo<D>::C];
  int bia[D][TYPES][SInfo<D>::Cb];
  int count;
};
template <int D, int NQ, int A>
constexpr WenoParityPoints<D, NQ, A> make_weno_parity_points() {
  using S = SInfo<D>;
  constexpr auto st = make_stencil_tables<D>();
  constexpr auto pt = make_parity_tables<D>();
  WenoParityPoints<D, NQ, A> w{};
  int k = 0;
  for (int s = 0; s < 2; s++)
    for (int z = 0; z < w.TYPES; z++)
      for (int p = 0; p < 1 << D; p++)  // class by class, as they are summed
        for (int n = 0; n < S::C; n++) {
          if (pt.neg[n] != p) continue;
          w.row[s][z][n] = (s == 0 || n < S::Cc) && !(p & parity_zero_axes(A, z)) ? k++ : -1;
        }
  for (int b = 0; b < D; b++)
    for (int z = 0; z < w.TYPES; z++)
      for (int p = 0; p < 1 << D; p++) {
        if (p >> b & 1) continue;
        for (int m = 0; m < S::Cb; m++) {
          const int zm = parity_zero_axes(A, z);
          if ((pt.neg[st.sub[2 * b][m]] & ~(1 << b)) != p) continue;
          w.bia[b][z][m] = -1;
          if (!(p & zm)) {
            w.bia[b][z][m] = k;
            k += zm >> b & 1 ? 1 : 2;
          }
        }
      }
  w.count = k;
  return w;
}

// Doubles of the whole list: derivatives, the D face axes, and with cells the
// interior points.
template <int D, int NQ>
constexpr int weno_parity_size(bool cells) {
  int n = make_weno_parity_deriv<D>().count + make_weno_parity_points<D, NQ, 0>().count +
          make_weno_parity_points<D, NQ, 1>().count;
  if (D == 3) n += make_weno_parity_points<D, NQ, D - 1>().count;
  if (cells) n += make_weno_parity_points<D, NQ, -1>().count;
  return n;
}

namespace detail {

// Coefficients of row e over the slots of the butterfly along the axes in mask.
template <int D>
void parity_expand(const double *e, int mask, double *c) {
  constexpr auto st = make_stencil_tables<D>();
  constexpr auto pt = make_parity_tables<D>();
  for (int n = 0; n < SInfo<D>::C; n++) {
    int nz = 0, pos = n;
    for (int d = 0; d < D; d++)
      if (mask >> d & 1) {
        if (st.off[n][d] != 0) nz |= 1 << d;
        if (st.off[n][d] < 0) pos = pt.mir[d][pos];
      }
    long double sum = 0.0L;
    int images = 0;
    for (int s = nz;; s = (s - 1) & nz) {
      int odd = 0, m = pos;
      for (int d = 0; d < D; d++)
        if (s >> d & 1) {
          m = pt.mir[d][m];
          odd ^= pt.neg[n] >> d & 1;
        }
      sum += (odd ? -1.0L : 1.0L) * (long double)e[m];
      images++;
      if (s == 0) break;
    }
    c[n] = double(sum / (long double)images);
  }
}

// Row of substencil s (0 full, 1 centre, then biased) over the full stencil's
// cells; mirrored along axis mir if >= 0.  False if it holds what no sum could.
template <int D>
bool substencil_row(const double *w, int s, int mir, double *e, double &big) {
  using S = SInfo<D>;
  constexpr auto st = make_stencil_tables<D>();
  constexpr auto pt = make_parity_tables<D>();
  std::fill(e, e + S::C, 0.0);
  big = 0.0;
  const int n = s == 0 ? S::C : (s == 1 ? S::Cc : S::Cb);
  for (int j = 0; j < n; j++) {
    const int m = s < 2 ? j : st.sub[s - 2][j];
    if (!std::isfinite(w[j])) return false;
    e[mir >= 0 ? pt.mir[mir][m] : m] = w[j];
    big = std::fmax(big, std::fabs(w[j]));
  }
  return true;
}

constexpr double parity_tol = 8.0 * 2.220446049250313e-16;  // of a row's largest weight

// Coefficients of the group's points from rows(s, point): row of substencil s.
template <int D, int NQ, int A, class Rows>
bool weno_parity_group(Rows rows, double *out) {
  using S = SInfo<D>;
  constexpr auto st = make_stencil_tables<D>();
  constexpr auto pt = make_parity_tables<D>();
  constexpr auto w = make_weno_parity_points<D, NQ, A>();
  constexpr int ALL = (1 << D) - 1;
  double e[S::C], c[S::C], ref[2][S::C], big;
  auto odd = [](int m) { return (m & 1) ^ (m >> 1 & 1) ^ (m >> 2 & 1); };
  for (int z = 0; z < w.TYPES; z++) {
    const int zm = parity_zero_axes(A, z);
    for (int s = 0; s < 2; s++)
      for (int sm = ALL; sm >= 0; sm--) {  // the point that is positive along sm, all-positive first
        if (sm & zm) continue;
        if (!substencil_row<D>(rows(s, parity_point(D, NQ, A, zm, sm)), s, -1, e, big)) return false;
        parity_expand<D>(e, ALL, c);
        if (sm == (ALL & ~zm)) std::copy(c, c + S::C, ref[0]);
        for (int n = 0; n < S::C; n++) {
          const double want = pt.neg[n] & zm ? 0.0 : (odd(pt.neg[n] & ~sm) ? -ref[0][n] : ref[0][n]);
          if (!(std::fabs(c[n] - want) <= parity_tol * big)) return false;
          if (sm == (ALL & ~zm) && w.row[s][z][n] >= 0) out[w.row[s][z][n]] = c[n];
        }
      }
    for (int b = 0; b < D; b++) {
      const int B = 1 << b;
      const bool zero = zm & B;
      for (int side = 0; side < 2; side++)
        for (int sm = ALL; sm >= 0; sm--) {
          if (sm & zm) continue;
          const int s = 2 + 2 * b + side;
          if (!substencil_row<D>(rows(s, parity_point(D, NQ, A, zm, sm)), s, side ? b : -1, e, big)) return false;
          parity_expand<D>(e, ALL & ~B, c);
          const int up = zero ? 0 : ((sm >> b & 1) ^ side);  // the mirrored side sees the mirrored point
          const bool first = side == 0 && (sm | B) == ((ALL & ~zm) | B);
          if (first) std::copy(c, c + S::C, ref[up]);
          for (int n = 0; n < S::C; n++) {
            const int neg = pt.neg[n] & ~B;
            const double want = neg & zm ? 0.0 : (odd(neg & ~sm) ? -ref[up][n] : ref[up][n]);
            if (!(std::fabs(c[n] - want) <= parity_tol * big)) return false;
          }
        }
      for (int m = 0; m < S::Cb; m++) {
        const int n = st.sub[2 * b][m], k = w.bia[b][z][m];
        const double f = st.off[n][b] != 0 ? 0.5 : 1.0;
        if (k < 0) continue;
        out[k] = zero ? f * ref[0][n] : 0.5 * f * (ref[1][n] + ref[0][n]);
        if (!zero) out[k + 1] = 0.5 * f * (ref[1][n] - ref[0][n]);
      }
    }
  }
  return true;
}

}  // namespace detail

// The whole list from the reference layouts face [nSub][2 D][Q][C], deriv
// [nSub][I][C] and, with cells, cell [nSub][NQ^D][C]; false when they lack the
// symmetry (tables set by the caller need not have it).
template <int D, int NQ>
bool weno_parity_list(const double *face, const double *deriv, const double *cell, std::vector<double> &out) {
  using S = SInfo<D>;
  constexpr auto st = make_stencil_tables<D>();
  constexpr auto w = make_weno_parity_deriv<D>();
  constexpr int Q = D == 3 ? NQ * NQ : NQ, NI = Q * NQ;
  out.assign(size_t(weno_parity_size<D, NQ>(cell != nullptr)), 0.0);
  double e[S::C], c[S::C], cp[S::C], big;
  for (int s = 0; s < S::nSub; s++) {
    // rows that are rounding noise beside the substencil's others are not held
    // to a symmetry of their own
    double all = 0.0;
    for (int i = 0; i < S::I; i++) {
      if (!detail::substencil_row<D>(deriv + (size_t(s) * S::I + i) * S::C, s, -1, e, big)) return false;
      all = std::fmax(all, big);
    }
    const int b = (s - 2) / 2;
    for (int i = 0; i < S::I; i++) {
      detail::substencil_row<D>(deriv + (size_t(s) * S::I + i) * S::C, s, -1, e, big);
      const double tol = detail::parity_tol * std::fmax(big, 2.2e-16 * all);
      if (s < 2) {
        detail::parity_expand<D>(e, (1 << D) - 1, c);
        for (int n = 0; n < S::C; n++) {
          const int k = w.row[s][i][n];
          if (k >= 0) out[k] = c[n];
          else if (!(std::fabs(c[n]) <= tol)) return false;
        }
      } else if (s % 2 == 0) {
        detail::parity_expand<D>(e, ((1 << D) - 1) & ~(1 << b), c);
        // the positive side's row is the mirror image up to its sign, which the square drops
        detail::substencil_row<D>(deriv + (size_t(s + 1) * S::I + i) * S::C, s + 1, b, e, big);
        detail::parity_expand<D>(e, ((1 << D) - 1) & ~(1 << b), cp);
        double same = 0.0, flip = 0.0;
        for (int n = 0; n < S::C; n++) {
          same = std::fmax(same, std::fabs(cp[n] - c[n]));
          flip = std::fmax(flip, std::fabs(cp[n] + c[n]));
        }
        if (!(std::fmin(same, flip) <= tol)) return false;
        for (int m = 0; m < S::Cb; m++) {
          const int n = st.sub[2 * b][m], k = w.bia[b][i][m];
          if (k >= 0) out[k] = (st.off[n][b] != 0 ? 0.5 : 1.0) * c[n];
          else if (!(std::fabs(c[n]) <= tol)) return false;
        }
      }
    }
  }
  auto rows = [&](int a) {
    return [=](int s, int p) { return face + ((size_t(s) * 2 * D + 2 * a) * Q + p) * S::C; };
  };
  double *o = out.data() + w.count;
  if (!detail::weno_parity_group<D, NQ, 0>(rows(0), o)) return false;
  o += make_weno_parity_points<D, NQ, 0>().count;
  if (!detail::weno_parity_group<D, NQ, 1>(rows(1), o)) return false;
  o += make_weno_parity_points<D, NQ, 1>().count;
  if (D == 3) {
    if (!detail::weno_parity_group<D, NQ, D - 1>(rows(D - 1), o)) return false;
    o += make_weno_parity_points<D, NQ, D - 1>().count;
  }
  if (cell)
    return detail::weno_parity_group<D, NQ, -1>([=](int s, int p) { return cell + (size_t(s) * NI + p) * S::C; }, o);
  return true;
}

}  // namespace kfvm
