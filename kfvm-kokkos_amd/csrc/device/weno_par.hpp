// KFVM-WENO in the mirror-symmetric form of host/parity_weno.hpp.
//
//   k_weno_par   Stencil_K.H:164-283, 416-454, 506-589: stencil values in
//                linearised primitive variables, smoothness indicators, WENO-AO
//                weights and the weighted face (GLM-MHD: and interior) states
#pragma once

namespace kfvm {
namespace dev {

template <int D>
struct WPTab {
  static constexpr WenoParityDeriv<D> W = make_weno_parity_deriv<D>();
};
template <int D, int NQ, int A>
struct WPPts {
  static constexpr WenoParityPoints<D, NQ, A> W = make_weno_parity_points<D, NQ, A>();
  // first coefficient of the group in the list
  static constexpr int base() {
    if constexpr (A == 0) return WPTab<D>::W.count;
    else if constexpr (A == -1) return WPPts<D, NQ, D - 1>::base() + WPPts<D, NQ, D - 1>::W.count;
    else return WPPts<D, NQ, A - 1>::base() + WPPts<D, NQ, A - 1>::W.count;
  }
};

// Byte offsets of the five cells around a cell along each axis, mapped into
// the grid, and the sides beyond which they lie (2 bits each: 1 low, 2 high;
// walls only).  The offset of a stencil cell is the sum of three of them.
template <int D>
struct StencilRef {
  unsigned o[3][5];
  unsigned side;
  __device__ __forceinline__ StencilRef(const Grid &g, int i, int j, int k) : side(0) {
#pragma unroll
    for (int d = 0; d < 5; d++) {
      int s;
      o[0][d] = unsigned(map_axis(i + d - 2, g.nx, g.bc[0], g.bc[1], s)) * 8u;
      side |= unsigned(s + 1) << (2 * d);
      o[1][d] = unsigned(map_axis(j + d - 2, g.ny, g.bc[2], g.bc[3], s)) * unsigned(g.nx) * 8u;
      side |= unsigned(s + 1) << (10 + 2 * d);
      if (D == 3) {
        o[2][d] = unsigned(map_axis(k + d - 2, g.nz, g.bc[4], g.bc[5], s)) * unsigned(g.nx) * unsigned(g.ny) * 8u;
        side |= unsigned(s + 1) << (20 + 2 * d);
      } else {
        o[2][d] = unsigned(k) * unsigned(g.nx) * unsigned(g.ny) * 8u;  // slice of a batch
      }
    }
  }
  // Values of variable w (one for the whole wave) over the stencil; the walls
  // negate those of the masks.
  __device__ __forceinline__ void load(const double *__restrict__ U, const Grid &g, int w,
                                       double (&q)[SInfo<D>::C]) const {
    const char *p = reinterpret_cast<const char *>(U + size_t(w) * g.ncell);
    // opaque, so that the sums are not kept in registers from one variable to the next
    unsigned x[5], y[5], z[5];
#pragma unroll
    for (int d = 0; d < 5; d++) {
      x[d] = o[0][d], y[d] = o[1][d], z[d] = o[2][D == 3 ? d : 2];
      asm volatile("" : "+v"(x[d]));
    }
    static_for<SInfo<D>::C>([&](auto nn) KFVM_INLINE {
      constexpr int n = decltype(nn)::value;
      constexpr int a = StTab<D>::ST.off[n][0] + 2, b = StTab<D>::ST.off[n][1] + 2, c = StTab<D>::ST.off[n][2] + 2;
      q[n] = *reinterpret_cast<const double *>(p + (x[a] + y[b] + z[c]));
    });
    // wall sides that negate w: bit 2 a + (0 low, 1 high)
    unsigned m = 0;
#pragma unroll
    for (int e = 0; e < 2 * D; e++) m |= ((g.negmask[e] >> w) & 1u) << e;
    if (m) {
      unsigned flip = 0;  // bit 5 a + d: the cells at that offset change sign
#pragma unroll
      for (int a = 0; a < D; a++)
#pragma unroll
        for (int d = 0; d < 5; d++) {
          const unsigned s = (side >> (10 * a + 2 * d)) & 3u;
          flip |= (((m >> (2 * a)) & s) ? 1u : 0u) << (5 * a + d);
        }
      static_for<SInfo<D>::C>([&](auto nn) KFVM_INLINE {
        constexpr int n = decltype(nn)::value;
        constexpr int x0 = StTab<D>::ST.off[n][0] + 2, y0 = StTab<D>::ST.off[n][1] + 7, z0 = StTab<D>::ST.off[n][2] + 12;
        unsigned b = (flip >> x0) ^ (flip >> y0);
        if (D == 3) b ^= flip >> z0;
        q[n] = __longlong_as_double(__double_as_longlong(q[n]) ^ ((unsigned long long)(b & 1u) << 63));
      });
    }
  }
};

// The biased substencils of axis B from the transformed values: those of the
// negative side (in the order of its cells) and of the positive side.  (The
// values are made opaque first: the sums of one call would otherwise be kept in
// registers for the next.)
template <int D, int B>
__device__ __forceinline__ void biased_values(double (&t)[SInfo<D>::C], double (&um)[SInfo<D>::Cb],
                                              double (&up)[SInfo<D>::Cb]) {
  static_for<SInfo<D>::Cb>([&](auto mm) KFVM_INLINE {
    constexpr int m = decltype(mm)::value, n = StTab<D>::ST.sub[2 * B][m];
    if constexpr (StTab<D>::ST.off[n][B] == 0) {
      um[m] = up[m] = t[n];
    } else {
      constexpr int p = PTab<D>::PT.mir[B][n];
      keep_here(t[p]);
      keep_here(t[n]);
      um[m] = t[p] - t[n];
      up[m] = t[p] + t[n];
    }
  });
}

// Smoothness indicators of all substencils.  A few rows at a time: the
// scheduler would fetch the coefficients of a whole substencil at once, more
// than the scalar registers hold.
template <int D>
__device__ __forceinline__ void parity_betas(double (&t)[SInfo<D>::C], const double *WP,
                                             double (&beta)[SInfo<D>::nSub]) {
  constexpr int C = SInfo<D>::C, Cb = SInfo<D>::Cb, I = SInfo<D>::I, RB = 4;
  static_for<2>([&](auto ss) KFVM_INLINE {
    constexpr int s = decltype(ss)::value;
    const double *w0 = WP;
    double b = 0.0;
    static_for<I>([&](auto ii) KFVM_INLINE {
      constexpr int i = decltype(ii)::value;
      if constexpr (i % RB == 0) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" : "+s"(w0));
      }
      const cdouble *w = (const cdouble *)w0;
      double acc = 0.0;
      static_for<C>([&](auto nn) KFVM_INLINE {
        constexpr int n = decltype(nn)::value, k = WPTab<D>::W.row[s][i][n];
        if constexpr (k >= 0) acc = fma(w[k], t[n], acc);
      });
      b = fma(acc, acc, b);
      keep_here(b);
    });
    beta[s] = b;
    __builtin_amdgcn_sched_barrier(0);
  });
  static_for<D>([&](auto bb) KFVM_INLINE {
    constexpr int B = decltype(bb)::value;
    const double *w0 = WP;
    double um[Cb], up[Cb];
    biased_values<D, B>(t, um, up);
    double bm = 0.0, bp = 0.0;
    static_for<I>([&](auto ii) KFVM_INLINE {
      constexpr int i = decltype(ii)::value;
      if constexpr (i % RB == 0) {
        __builtin_amdgcn_sched_barrier(0);
        asm volatile("" : "+s"(w0));
      }
      const cdouble *w = (const cdouble *)w0;
      double am = 0.0, ap = 0.0;
      static_for<Cb>([&](auto mm) KFVM_INLINE {
        constexpr int m = decltype(mm)::value, k = WPTab<D>::W.bia[B][i][m];
        if constexpr (k >= 0) {
          am = fma(w[k], um[m], am);
          ap = fma(w[k], up[m], ap);
        }
      });
      bm = fma(am, am, bm);
      bp = fma(ap, ap, bp);
      keep_here(bm);
      keep_here(bp);
    });
    beta[2 + 2 * B] = bm;
    beta[3 + 2 * B] = bp;
    __builtin_amdgcn_sched_barrier(0);
  });
}

// Weighted values at the points of group A: every substencil's parts go into
// the parity classes e[type][class] of the points, one butterfly ends it.
template <int D, int NQ, int A>
__device__ __forceinline__ void weno_points(double (&t)[SInfo<D>::C], const double *WP,
                                            const double (&om)[SInfo<D>::nSub],
                                            double (&out)[ParPts<D, NQ, A>::N]) {
  constexpr int C = SInfo<D>::C, Cb = SInfo<D>::Cb, ALL = (1 << D) - 1, TYPES = ParPts<D, NQ, A>::TYPES;
  using P = WPPts<D, NQ, A>;
  double e[TYPES][ALL + 1];
  const double *w0 = WP + P::base();
  asm volatile("" : "+s"(w0));
  static_for<TYPES>([&](auto zz) KFVM_INLINE {
    constexpr int z = decltype(zz)::value, zm = parity_zero_axes(A, z);
    const cdouble *w = (const cdouble *)w0;
    static_for<ALL + 1>([&](auto pp) KFVM_INLINE {
      constexpr int p = decltype(pp)::value;
      if constexpr (!(p & zm)) {
        double f = 0.0, c = 0.0;
        static_for<C>([&](auto nn) KFVM_INLINE {
          constexpr int n = decltype(nn)::value;
          if constexpr (PTab<D>::PT.neg[n] == p) {
            constexpr int k = P::W.row[0][z][n], kc = P::W.row[1][z][n];
            f = fma(w[k], t[n], f);
            if constexpr (kc >= 0) c = fma(w[kc], t[n], c);
          }
        });
        e[z][p] = fma(om[1], c, om[0] * f);
      }
    });
  });
  __builtin_amdgcn_sched_barrier(0);
  static_for<D>([&](auto bb) KFVM_INLINE {
    constexpr int B = decltype(bb)::value, BB = 1 << B;
    const double *w1 = w0;
    asm volatile("" : "+s"(w1));
    const cdouble *w = (const cdouble *)w1;
    double um[Cb], up[Cb];
    biased_values<D, B>(t, um, up);
    const double oM = om[2 + 2 * B], oP = om[3 + 2 * B];
    static_for<TYPES>([&](auto zz) KFVM_INLINE {
      constexpr int z = decltype(zz)::value, zm = parity_zero_axes(A, z);
      static_for<ALL + 1>([&](auto pp) KFVM_INLINE {
        constexpr int p = decltype(pp)::value;
        if constexpr (!(p & zm) && !(p & BB)) {
          double em = 0.0, ep = 0.0, dm = 0.0, dp = 0.0;
          static_for<Cb>([&](auto mm) KFVM_INLINE {
            constexpr int m = decltype(mm)::value, n = StTab<D>::ST.sub[2 * B][m], k = P::W.bia[B][z][m];
            if constexpr ((PTab<D>::PT.neg[n] & ~BB) == p) {
              em = fma(w[k], um[m], em);
              ep = fma(w[k], up[m], ep);
              if constexpr (!(zm & BB)) {
                dm = fma(w[k + 1], um[m], dm);
                dp = fma(w[k + 1], up[m], dp);
              }
            }
          });
          e[z][p] = fma(oP, ep, fma(oM, em, e[z][p]));
          if constexpr (!(zm & BB)) e[z][p | BB] = fma(-oP, dp, fma(oM, dm, e[z][p | BB]));
        }
      });
    });
    __builtin_amdgcn_sched_barrier(0);
  });
  static_for<TYPES>([&](auto zz) KFVM_INLINE {
    constexpr int z = decltype(zz)::value, zm = parity_zero_axes(A, z);
    static_for<D>([&](auto dd) KFVM_INLINE {
      static_for<ALL + 1>([&](auto pp) KFVM_INLINE {
        constexpr int d = decltype(dd)::value, p = decltype(pp)::value;
        if constexpr (!(zm >> d & 1) && !(p >> d & 1) && !(p & zm)) {
          const double ev = e[z][p], od = e[z][p | (1 << d)];
          e[z][p] = ev - od;
          e[z][p | (1 << d)] = ev + od;
        }
      });
    });
    static_for<ALL + 1>([&](auto ss) KFVM_INLINE {
      constexpr int s = decltype(ss)::value;
      if constexpr (!(s & zm)) {
        keep_here(e[z][s]);
        out[parity_point(D, NQ, A, zm, s)] = e[z][s];
      }
    });
  });
}

// One wave takes 64 listed cells (all cells without a list) and one variable,
// so the variable's branch of the conversion is uniform; a workgroup's waves are
// the variables of the same cells.  Each wave gathers its own variable once and
// hands it to the others, whose conversion needs it, through LDS.  (With the
// pressure's wave gathering the other variables itself, that wave's five or nine
// rounds of latency kept 1.2 waves busy per SIMD.)  Euler rows (WS, for list
// positions below cap) leave through LDS, so that whole rows are written.
// Per cell and variable the 3D 2x2 rule takes about 1900 FP64 operations instead
// of the 4600 products of the dense form, from a 6 KB coefficient list that
// stays in the scalar cache.  The 67 KB (GLM-MHD: 135 KB) of handed-over values
// bound it to ten (nine) waves a CU.  Dense / this kernel, ms per evaluation:
// Euler 160 x 144 x 152 (15 % of the cells) 1.14 / 0.64, 64^3 0.151 / 0.084, 75 x
// 62 x 81 with the 3x3 rule 0.267 / 0.113, 2D batch of 48 x 128^2 0.055 / 0.031,
// GLM-MHD 96^3 with the limiter's pass 1.07 / 0.74.
template <int D, int NQ, int NV>
struct WenoPar {
  static constexpr int N = ParPts<D, NQ, 0>::N, FQ = D * N;
  static constexpr int NT = 64 * NV;
  static constexpr int ROW = N * NV + 1;  // LDS row of one cell and face axis, padded against bank conflicts
  static constexpr int VALS = (NV - 1) * SInfo<D>::C * 64;  // stencil values of all variables but the energy
  // POST: whole rows of the cells in LDS, then lanes per cell for the limiter
  static constexpr int ROWF = FQ * NV + 1, G = 4;
  static constexpr int lds(bool post) {
    const int r = NV != 5 ? 0 : 64 * (post ? ROWF : ROW);
    return r > VALS ? r : VALS;
  }
  // 3D 3x3: 18 accumulators and their points need the 256 registers of two waves per SIMD
  static constexpr int WAVES = D == 3 && NQ == 3 ? 2 : 3;
};

// POST (Euler, every listed cell has a row): the workgroup also does k_weno_post's
// work on its cells while their rows are in LDS, so that they cross HBM once:
// 160 x 144 x 152 0.68 ms for both instead of 0.46 + 0.30, 64^3 87 us instead of
// 62 + 29 and a launch.
template <int D, int NQ, int NV, bool POST>
__global__ __launch_bounds__((WenoPar<D, NQ, NV>::NT), (WenoPar<D, NQ, NV>::WAVES)) void k_weno_par(
    const double *__restrict__ U, double *__restrict__ FS, double *__restrict__ SRC, Grid g,
    const double *__restrict__ WP, const int *__restrict__ list, const int *__restrict__ counter,
    double *__restrict__ WS, int cap, double *__restrict__ thetaNew, const double *__restrict__ props) {
  using K = WenoPar<D, NQ, NV>;
  constexpr int C = SInfo<D>::C, nSub = SInfo<D>::nSub, N = K::N, FQ = K::FQ;
  constexpr double gHi = 0.7, gLo = 0.7;
  constexpr double g0 = gHi, g1 = (1.0 - gHi) * gLo, gb = (1.0 - gHi) * (1.0 - gLo) / double(2 * D);
  __shared__ double lds[K::lds(POST)];
  const int n = list ? *counter : g.ncell;
  const int lane = threadIdx.x & 63;
  const int v = __builtin_amdgcn_readfirstlane(int(threadIdx.x) >> 6);
  const size_t nc = g.ncell;
#pragma unroll 1
  for (int t0 = blockIdx.x * 64; t0 < n; t0 += gridDim.x * 64) {
    const bool live = t0 + lane < n;
    const int c = live ? (list ? list[t0 + lane] : t0 + lane) : (list ? list[t0] : t0);
    double t[C];
    {
      // opaque: what derives from the grid is cheap on the scalar unit and would
      // otherwise be kept, spilled, from one group of cells to the next
      Grid gl = g;
      asm volatile("" : "+s"(gl.nx), "+s"(gl.ny), "+s"(gl.nz));
#pragma unroll
      for (int e = 0; e < 2 * D; e++) asm volatile("" : "+s"(gl.bc[e]), "+s"(gl.negmask[e]));
      int i, j, k;
      cell_ijk<D>(c, gl, i, j, k);
      const StencilRef<D> sr(gl, i, j, k);
      sr.load(U, gl, v, t);
      __syncthreads();  // the last cells' values and rows have been read
      if (v != 4) {
        double *d = lds + (v < 4 ? v : v - 1) * (C * 64) + lane;
#pragma unroll
        for (int m = 0; m < C; m++) d[m * 64] = t[m];
      }
      __syncthreads();
      // linearised primitive variables (VarConvert): velocities (m - u rho) /
      // rho_c, pressure (gamma - 1)(E + q^2/2 rho - u.m - B_c.B - psi_c psi)
      constexpr int m0 = detail::find_idx<D>(StTab<D>::ST, 0, 0, 0), L0 = m0 * 64;  // the cell itself
      if (v >= 1 && v <= 3) {
        const double rho = lds[L0 + lane], ir = 1.0 / rho, u = t[m0] / rho;
#pragma unroll
        for (int m = 0; m < C; m++) t[m] = (t[m] - u * lds[m * 64 + lane]) * ir;
      } else if (v == 4) {
        const double rho = lds[L0 + lane];
#pragma unroll 1
        for (int x = 0; x < NV - 1; x++) {
          const double *q = lds + x * (C * 64) + lane;
          double cw;
          if (x == 0) {
            const double a = q[C * 64 + L0] / rho, b = q[2 * C * 64 + L0] / rho, e = q[3 * C * 64 + L0] / rho;
            cw = (a * a + b * b + e * e) / 2.0;
          } else {
            cw = x < 4 ? -(q[L0] / rho) : -q[L0];
          }
#pragma unroll
          for (int m = 0; m < C; m++) t[m] = fma(cw, q[m * 64], t[m]);
        }
#pragma unroll
        for (int m = 0; m < C; m++) t[m] *= g.gamma - 1.0;
      }
    }
    parity_transform<D>(t);
    __builtin_amdgcn_sched_barrier(0);
    double om[nSub];
    parity_betas<D>(t, WP, om);
    double tot = 0.0;
#pragma unroll
    for (int s = 0; s < nSub; s++) {
      const double gs = s == 0 ? g0 : (s == 1 ? g1 : gb);
      om[s] = gs / (om[s] * om[s] + 1.e-40);
      tot += om[s];
    }
#pragma unroll
    for (int s = 0; s < nSub; s++) om[s] /= tot;
    om[0] /= g0;
#pragma unroll
    for (int s = 1; s < nSub; s++) om[s] -= om[0] * (s == 1 ? g1 : gb);
    __builtin_amdgcn_sched_barrier(0);
    static_for<D>([&](auto aa) KFVM_INLINE {
      constexpr int A = decltype(aa)::value;
      double out[N];
      weno_points<D, NQ, A>(t, WP, om, out);
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (POST) {
        if (A == 0) __syncthreads();  // what the rows overwrite has been read
#pragma unroll
        for (int p = 0; p < N; p++) lds[lane * K::ROWF + (A * N + p) * NV + v] = out[p];
      } else if constexpr (NV == 5) {
        if (list) {
          __syncthreads();  // what the rows overwrite has been read
#pragma unroll
          for (int p = 0; p < N; p++) lds[lane * K::ROW + p * NV + v] = out[p];
          __syncthreads();
          const int rows = (n < cap ? n : cap) - t0;
          for (int x = threadIdx.x; x < 64 * N * NV; x += K::NT) {
            const int r = x / (N * NV), q = x % (N * NV);
            if (r < rows) WS[size_t(t0 + r) * (FQ * NV) + A * N * NV + q] = lds[r * K::ROW + q];
          }
        }
        if (live && !(list && t0 + lane < cap)) {
          double *d = FS + fs_base(c, FQ * NV) + size_t(A * N * NV + v) * FSB;
#pragma unroll
          for (int p = 0; p < N; p++) d[size_t(p * NV) * FSB] = out[p];
        }
      } else if (live) {
        double *d = FS + fs_base(c, FQ * NV) + size_t(A * N * NV + v) * FSB;
#pragma unroll
        for (int p = 0; p < N; p++) d[size_t(p * NV) * FSB] = out[p];
      }
    });
    if constexpr (POST) {
      __syncthreads();
      const int m = threadIdx.x / K::G;
      if (m < 64 && t0 + m < n) {  // whole groups of lanes
        const int cell = list[t0 + m], pl = threadIdx.x % K::G;
        const double th = weno_post_cell<D, NQ, K::G>(lds + m * K::ROWF, 1, U, props, g, cell, pl);
        if (pl == 0) thetaNew[cell] = th;
      }
      __syncthreads();
      const int rows = n - t0 < 64 ? n - t0 : 64;
      for (int x = threadIdx.x; x < rows * FQ * NV; x += K::NT)
        WS[size_t(t0) * (FQ * NV) + x] = lds[x / (FQ * NV) * K::ROWF + x % (FQ * NV)];
    }
    if constexpr (NV == 9) {
      constexpr int NI = ParPts<D, NQ, -1>::N;
      double out[NI];
      weno_points<D, NQ, -1>(t, WP, om, out);
      if (live) {
#pragma unroll
        for (int p = 0; p < NI; p++) SRC[(size_t(p) * NV + v) * nc + c] = out[p];
      }
    }
  }
}

}  // namespace dev
}  // namespace kfvm
