// The mirror-symmetric WENO list (parity_weno.hpp) evaluated as the kernel does,
// against the dense rows it was made from: every substencil's derivatives and
// points, for every rule; then tables without the symmetry, which it refuses.
#include <cmath>
#include <cstdio>
#include <cstdlib>

#include "parity_weno.hpp"
#include "weights.hpp"

using namespace kfvm;

static int bad = 0;
static double worst = 0.0;
// difference in units of its bound: each side sums at most 33 products and 60
// sums of rounded values, 128 eps of the sum of magnitudes
static void compare(double a, double b, double mag) {
  const double r = std::fabs(a - b) / (128 * 2.220446049250313e-16 * mag);
  worst = std::fmax(worst, r);
  if (!(r <= 1.0)) bad++;
}

template <int D, int NQ, int A>
static void points(const double *w, const double *t, const double *x, const double *rows, size_t perSub) {
  using S = SInfo<D>;
  constexpr auto st = make_stencil_tables<D>();
  constexpr auto pt = make_parity_tables<D>();
  constexpr auto W = make_weno_parity_points<D, NQ, A>();
  constexpr int ALL = (1 << D) - 1;
  for (int s = 0; s < S::nSub; s++)
    for (int z = 0; z < W.TYPES; z++) {
      const int zm = parity_zero_axes(A, z), b = (s - 2) / 2;
      double e[ALL + 1] = {};
      if (s < 2) {
        for (int n = 0; n < S::C; n++)
          if (W.row[s][z][n] >= 0) e[pt.neg[n]] += w[W.row[s][z][n]] * t[n];
      } else {
        for (int m = 0; m < S::Cb; m++) {
          const int n = st.sub[2 * b][m], k = W.bia[b][z][m], p = pt.neg[n] & ~(1 << b);
          if (k < 0) continue;
          const int q = pt.mir[b][n];
          const double u = st.off[n][b] == 0 ? t[n] : (s % 2 ? t[q] + t[n] : t[q] - t[n]);
          e[p] += w[k] * u;
          if (!(zm >> b & 1)) e[p | 1 << b] += (s % 2 ? -w[k + 1] : w[k + 1]) * u;
        }
      }
      for (int sm = 0; sm <= ALL; sm++) {  // the point positive along sm
        if (sm & zm) continue;
        double v = 0.0;
        for (int p = 0; p <= ALL; p++) v += (__builtin_popcount(p & ~sm) & 1 ? -e[p] : e[p]);
        const double *r = rows + size_t(s) * perSub + size_t(parity_point(D, NQ, A, zm, sm)) * S::C;
        double d = 0.0, mag = 0.0;
        const int cnt = s == 0 ? S::C : (s == 1 ? S::Cc : S::Cb);
        for (int j = 0; j < cnt; j++) {
          const double y = x[s < 2 ? j : st.sub[s - 2][j]];
          d += r[j] * y;
          mag += std::fabs(r[j] * y);
        }
        compare(v, d, mag);
      }
    }
}

template <int D, int NQ>
static void rule() {
  using S = SInfo<D>;
  constexpr auto st = make_stencil_tables<D>();
  constexpr auto pt = make_parity_tables<D>();
  constexpr auto W = make_weno_parity_deriv<D>();
  constexpr int Q = D == 3 ? NQ * NQ : NQ;
  WeightTable T = build_weights(D, NQ, 5.0, 0.01, 0.013, 0.017);
  std::vector<double> o;
  if (!weno_parity_list<D, NQ>(T.face.data(), T.deriv.data(), T.cell.data(), o)) {
    std::printf("refused: dim %d nq %d\n", D, NQ);
    bad++;
    return;
  }
  double x[S::C], t[S::C];
  for (int n = 0; n < S::C; n++) t[n] = x[n] = 0.5 + std::rand() / double(RAND_MAX);
  for (int d = 0; d < D; d++)
    for (int n = 0; n < S::C; n++)
      if (st.off[n][d] > 0) {
        const int m = pt.mir[d][n];
        const double s = t[n] + t[m], f = t[n] - t[m];
        t[n] = s;
        t[m] = f;
      }
  for (int s = 0; s < S::nSub; s++)
    for (int i = 0; i < S::I; i++) {
      const int b = (s - 2) / 2, cnt = s == 0 ? S::C : (s == 1 ? S::Cc : S::Cb);
      double d = 0.0, mag = 0.0, v = 0.0, big = 0.0;
      for (int j = 0; j < cnt; j++) {
        const double y = x[s < 2 ? j : st.sub[s - 2][j]];
        d += T.d(s, i, j) * y;
        mag += std::fabs(T.d(s, i, j) * y);
      }
      for (int r = 0; r < S::I; r++)
        for (int j = 0; j < cnt; j++) big = std::fmax(big, std::fabs(T.d(s, r, j)));
      for (int n = 0; s < 2 && n < S::C; n++)
        if (W.row[s][i][n] >= 0) v += o[W.row[s][i][n]] * t[n];
      for (int m = 0; s >= 2 && m < S::Cb; m++) {
        const int n = st.sub[2 * b][m], k = W.bia[b][i][m], q = pt.mir[b][n];
        if (k >= 0) v += o[k] * (st.off[n][b] == 0 ? t[n] : (s % 2 ? t[q] + t[n] : t[q] - t[n]));
      }
      // the square drops the sign; rows that are rounding noise beside the others count as zero
      compare(std::fabs(v), std::fabs(d), mag + 2.2e-16 * big);
    }
  const double *w = o.data() + W.count;
  points<D, NQ, 0>(w, t, x, T.face.data(), size_t(2 * D) * Q * S::C);
  w += make_weno_parity_points<D, NQ, 0>().count;
  points<D, NQ, 1>(w, t, x, T.face.data() + size_t(2) * Q * S::C, size_t(2 * D) * Q * S::C);
  w += make_weno_parity_points<D, NQ, 1>().count;
  if (D == 3) {
    points<D, NQ, D - 1>(w, t, x, T.face.data() + size_t(2 * (D - 1)) * Q * S::C, size_t(2 * D) * Q * S::C);
    w += make_weno_parity_points<D, NQ, D - 1>().count;
  }
  points<D, NQ, -1>(w, t, x, T.cell.data(), size_t(Q) * NQ * S::C);
  // one changed weight anywhere: refused
  for (int which = 0; which < 3; which++) {
    WeightTable B = T;
    std::vector<double> &tab = which == 0 ? B.face : (which == 1 ? B.deriv : B.cell);
    size_t at = 0;
    for (size_t e = 0; e < tab.size(); e++)
      if (std::fabs(tab[e]) > std::fabs(tab[at])) at = e;
    tab[at] *= 1.0 + 1e-12;
    if (weno_parity_list<D, NQ>(B.face.data(), B.deriv.data(), B.cell.data(), o)) {
      std::printf("accepted a table without the symmetry: dim %d nq %d, table %d\n", D, NQ, which);
      bad++;
    }
  }
}

int main() {
  rule<2, 2>();
  rule<2, 3>();
  rule<3, 2>();
  rule<3, 3>();
  std::printf("worst %.3f of the bound, %d failures\n", worst, bad);
  return bad != 0;
}
