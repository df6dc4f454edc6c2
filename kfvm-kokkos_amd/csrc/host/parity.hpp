// Mirror-symmetric form of the full-stencil reconstruction weights.
//
// The radius-2 stencil and the Gauss points are symmetric under the mirror of
// every axis, and so are the full-stencil weights: the weight of cell o for
// point p equals that of the mirrored cell for the mirrored point.  The dot
// products of all mirror images of a point therefore split into parity
// classes (one bit per axis: even or odd in that axis).  With
//   T[n]  the stencil values after one sum / difference butterfly per axis
//         (in place: the cell on the positive side of the axis takes the sum,
//         its mirror image the difference), so slot n holds the combination
//         of the mirror images of |o_n| that is odd in the axes where o_n < 0,
//   c[n]  the matching combination of the weights of the point whose nonzero
//         coordinates are all positive, divided by the number of images,
// the sum of c[n] T[n] over the slots of class p is the part of the dot product
// that is odd in the axes of p, and a second butterfly over the classes gives
// the value at every mirror image of the point.  In 3D the 24 face points of a
// 2x2 rule take 3 x (33 products and sums + 24 sums) after 60 shared sums
// instead of 24 x 33 products; the sums run in another order than the dense dot
// product, so results agree to rounding.
//
// The weights of the three face axes are one set up to a permutation of the
// axes (they are set up in cells, whatever dx, dy, dz; the y and z faces' are
// mapped from the x faces'), so one list of coefficients, that of the x axis,
// serves all of them (parity_frame_axis: the permutation).
#pragma once

#include <cmath>
#include <vector>

#include "stencil_geom.hpp"

namespace kfvm {

template <int D>
struct ParityTables {
  int neg[SInfo<D>::C];     // axes (bits) in which slot n is odd: those with offset < 0
  int mir[3][SInfo<D>::C];  // mirror image of cell n along an axis
  bool first[SInfo<D>::C];  // slot n is the first of its class
};

template <int D>
constexpr ParityTables<D> make_parity_tables() {
  ParityTables<D> p{};
  constexpr auto t = make_stencil_tables<D>();
  for (int n = 0; n < SInfo<D>::C; n++) {
    p.neg[n] = 0;
    for (int d = 0; d < D; d++) {
      if (t.off[n][d] < 0) p.neg[n] |= 1 << d;
      p.mir[d][n] = detail::find_idx<D>(t, d == 0 ? -t.off[n][0] : t.off[n][0],
                                        d == 1 ? -t.off[n][1] : t.off[n][1], d == 2 ? -t.off[n][2] : t.off[n][2]);
    }
    p.first[n] = true;
    for (int m = 0; m < n; m++)
      if (p.neg[m] == p.neg[n]) p.first[n] = false;
  }
  return p;
}

// Point types of one face axis: which transverse axes have coordinate zero
// (only the 3-point rule has such nodes), and of the interior points: which
// axes have.  Bit b of a type is the b-th transverse axis (ascending), or the
// axis itself for interior points.
KFVM_HD constexpr int parity_face_types(int dim, int nq) { return nq == 3 ? 1 << (dim - 1) : 1; }
KFVM_HD constexpr int parity_cell_types(int dim, int nq) { return nq == 3 ? 1 << dim : 1; }

// Axis of the grid that plays the role of axis r (0: normal, 1, 2: transverse)
// of the x faces for face axis a; interior points (a = -1) are not permuted.
KFVM_HD constexpr int parity_frame_axis(int a, int r) {
  return a <= 0 ? r : (r == 0 ? a : (a == 1 ? (r == 1 ? 0 : 2) : (r == 1 ? 1 : 0)));
}

// Axes (bits) along which the points of type z are zero.
KFVM_HD constexpr int parity_zero_axes(int a, int z) {
  if (a < 0) return z;
  return ((z & 1) << parity_frame_axis(a, 1)) | ((z >> 1 & 1) << parity_frame_axis(a, 2));
}

// Slot of face axis a's stencil that corresponds to slot m of the x axis'.
template <int D>
constexpr int parity_slot(int a, int m) {
  const auto t = make_stencil_tables<D>();
  int o[3] = {0, 0, 0};
  for (int r = 0; r < D; r++) o[parity_frame_axis(a, r)] = t.off[m][r];
  return detail::find_idx<D>(t, o[0], o[1], o[2]);
}
template <int D>
struct ParitySlots {
  int slot[3][SInfo<D>::C];
};
template <int D>
constexpr ParitySlots<D> make_parity_slots() {
  ParitySlots<D> r{};
  for (int a = 0; a < D; a++)
    for (int m = 0; m < SInfo<D>::C; m++) r.slot[a][m] = parity_slot<D>(a, m);
  return r;
}

// Node index of a coordinate: the 2-point rule orders its nodes {-, +}, the
// 3-point rule {0, -, +} (quad_rule).
KFVM_HD constexpr int parity_node(int nq, bool zero, bool positive) {
  return nq == 2 ? (positive ? 1 : 0) : (zero ? 0 : (positive ? 2 : 1));
}

// Point index, within the 2 Q points of face axis a (lower face first) or the
// NQ^D interior points (a = -1), of the point that is zero along the axes of
// zmask and positive along those of smask.
KFVM_HD constexpr int parity_point(int dim, int nq, int a, int zmask, int smask) {
  int q = 0;
  for (int d = 0; d < dim; d++)
    if (d != a) q = q * nq + parity_node(nq, (zmask >> d) & 1, (smask >> d) & 1);
  int Q = 1;
  for (int d = 1; d < dim; d++) Q *= nq;
  return a < 0 ? q : ((smask >> a) & 1) * Q + q;
}

// The coefficients c of every point type from the dense rows of the points,
// rows[point][C] (point as parity_point numbers them): out[type][C], in the
// slots of the x axis.  False when the rows are not mirror-symmetric to
// rounding (tables set by the caller need not be).
template <int D>
bool parity_coefficients(int nq, int a, const double *rows, double *out) {
  constexpr int C = SInfo<D>::C;
  const auto st = make_stencil_tables<D>();
  const auto pt = make_parity_tables<D>();
  const int types = a >= 0 ? parity_face_types(D, nq) : parity_cell_types(D, nq);
  const int all = (1 << D) - 1;
  // image of cell n under the mirrors of the axes in m
  auto image = [&](int n, int m) {
    for (int d = 0; d < D; d++)
      if ((m >> d) & 1) n = pt.mir[d][n];
    return n;
  };
  for (int z = 0; z < types; z++) {
    const int zm = parity_zero_axes(a, z);
    const double *rep = rows + size_t(parity_point(D, nq, a, zm, all & ~zm)) * C;
    double big = 0.0;
    for (int n = 0; n < C; n++) {
      if (!std::isfinite(rep[n])) return false;
      big = std::fmax(big, std::fabs(rep[n]));
    }
    const double tol = 8.0 * 2.220446049250313e-16 * big;
    for (int s = 0; s <= all; s++) {  // mirrors of the point, and those that leave it in place
      const double *r = rows + size_t(parity_point(D, nq, a, zm, (all & ~zm) & ~s)) * C;
      for (int n = 0; n < C; n++)
        if (!(std::fabs(r[image(n, s)] - rep[n]) <= tol)) return false;
    }
    for (int m = 0; m < C; m++) {
      const int n = a > 0 ? parity_slot<D>(a, m) : m;
      int nz = 0, pos = n;
      for (int d = 0; d < D; d++) {
        if (st.off[n][d] != 0) nz |= 1 << d;
        if (st.off[n][d] < 0) pos = pt.mir[d][pos];
      }
      long double sum = 0.0L;
      int images = 0;
      for (int s = nz;; s = (s - 1) & nz) {  // every subset of the nonzero axes mirrored
        int odd = 0;
        for (int d = 0; d < D; d++)
          if ((s & pt.neg[n]) >> d & 1) odd ^= 1;
        sum += (odd ? -1.0L : 1.0L) * (long double)rep[image(pos, s)];
        images++;
        if (s == 0) break;
      }
      out[size_t(z) * C + m] = double(sum / (long double)images);
    }
  }
  return true;
}

// The one coefficient list of all face axes, out[type][C], from the
// full-stencil rows face[2 D][Q][C]; false when they lack the symmetry.
template <int D>
bool parity_face_list(int nq, const double *face, std::vector<double> &out) {
  constexpr int C = SInfo<D>::C;
  const int types = parity_face_types(D, nq), Q = D == 3 ? nq * nq : nq;
  out.assign(size_t(types) * C, 0.0);
  std::vector<double> c(out.size());
  for (int a = 0; a < D; a++) {
    if (!parity_coefficients<D>(nq, a, face + size_t(2 * a) * Q * C, a == 0 ? out.data() : c.data())) return false;
    for (int z = 0; z < types && a > 0; z++) {
      double big = 0.0;
      for (int n = 0; n < C; n++) big = std::fmax(big, std::fabs(out[size_t(z) * C + n]));
      for (int n = 0; n < C; n++)
        if (!(std::fabs(c[size_t(z) * C + n] - out[size_t(z) * C + n]) <= 8.0 * 2.220446049250313e-16 * big))
          return false;
    }
  }
  return true;
}

}  // namespace kfvm
