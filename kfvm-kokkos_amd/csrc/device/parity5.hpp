// Full-stencil reconstruction in its mirror-symmetric (parity) form, and the
// fused sparse-mode path of the Euler (5-variable) equations built on it.
//
//   parity_transform, parity_points   Stencil_K.H:32-90 in the form of
//                 host/parity.hpp: one butterfly over the stencil values of a
//                 variable, then 33 (2D: 13) products per face axis for all of
//                 its points.
//   k_linear_par  the linear pass: face states of every cell (to FS, or only
//                 those on brick boundaries), the Numeric_K.H:315-379 indicator
//                 and the Common_K.H:299-643 limiter's fast test.
//   k_pp_rows     Common_K.H:299-643: the limiter's exact sequence for the
//                 cells whose linear states failed the fast test of the linear
//                 pass (and that the selector did not hand to WENO); their
//                 limited states go to a compact row, like the WENO cells'.
//   k_flux_par    linear face states of every cell that has no row, recomputed
//                 from the brick staged in LDS, then Common_K.H:180-297 Riemann
//                 solves, Numeric_K.H:109-196 flux divergence and
//                 Numeric_K.H:198-290 RK register update and error norm.
//
// Storing every face state (16 GB at 256^3 per stage, written and read back)
// costs the unfused pair of kernels more than recomputing the states in the
// parity form, so only the brick-boundary planes (3 GB) and the rows of WENO /
// limited cells cross HBM.  Linear pass + flux kernel, ms (fused / both kernels
// unfused with parity linear states / dense linear states): 64^3 0.20 / 0.28 /
// 0.31, 160 x 144 x 152 2.59 / 2.62 / 2.92, 2D 1024^2 (learned selection) 0.21 /
// 0.31 / 0.32.  (With pow_pos in place of the library function the fused pair takes
// 0.18 at 64^3 and 2.21 at 160 x 144 x 152.)
#pragma once

namespace kfvm {
namespace dev {

template <int D>
struct PTab {
  static constexpr ParityTables<D> PT = make_parity_tables<D>();
  static constexpr ParitySlots<D> SL = make_parity_slots<D>();
};

// Calls f(integral_constant<I>) for I = 0 .. N - 1: a loop whose index is a
// constant expression.  (Nests of this size with table look-ups exceed what the
// loop unroller folds, and what it leaves indexes registers at run time.)
template <class F, int... I>
__device__ __forceinline__ void static_for_seq(F &&f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}
template <int N, class F>
__device__ __forceinline__ void static_for(F &&f) {
  static_for_seq(f, std::make_integer_sequence<int, N>{});
}
#define KFVM_INLINE __attribute__((always_inline))

// The value is formed here: the compiler would otherwise sink a sum, a test or a
// maximum to its last use and keep all its terms in registers until then (724 B
// of scratch a thread instead of none in 3D).
__device__ __forceinline__ void keep_here(double &x) { asm volatile("" : "+v"(x)); }
__device__ __forceinline__ void keep_here(int &x) { asm volatile("" : "+v"(x)); }

// The butterflies over the stencil values of one variable, in place.
template <int D>
__device__ __forceinline__ void parity_transform(double (&t)[SInfo<D>::C]) {
  static_for<D>([&](auto dd) KFVM_INLINE {
    static_for<SInfo<D>::C>([&](auto nn) KFVM_INLINE {
      constexpr int d = decltype(dd)::value, n = decltype(nn)::value;
      if constexpr (StTab<D>::ST.off[n][d] > 0) {
        constexpr int m = PTab<D>::PT.mir[d][n];
        const double s = t[n] + t[m], f = t[n] - t[m];
        t[n] = s;
        t[m] = f;
      }
    });
  });
}

// Number of points parity_points produces: both faces of axis A, or the
// interior points (A = -1).
template <int D, int NQ, int A>
struct ParPts {
  static constexpr int Q = D == 3 ? NQ * NQ : NQ;
  static constexpr int N = A >= 0 ? 2 * Q : Q * NQ;
  static constexpr int TYPES = A >= 0 ? parity_face_types(D, NQ) : parity_cell_types(D, NQ);
};

// Values at the points of face axis A (lower face's Q points, then the upper
// face's), or at the interior points (A = -1), from the transformed stencil
// values t and the coefficients w[type][C] (one list for every face axis).
template <int D, int NQ, int A, class WP>
__device__ __forceinline__ void parity_points(const double (&t)[SInfo<D>::C], WP w,
                                              double (&out)[ParPts<D, NQ, A>::N]) {
  constexpr int C = SInfo<D>::C, ALL = (1 << D) - 1;
  static_for<ParPts<D, NQ, A>::TYPES>([&](auto zz) KFVM_INLINE {
    constexpr int z = decltype(zz)::value, zm = parity_zero_axes(A, z);
    double e[ALL + 1];
#pragma unroll
    for (int p = 0; p <= ALL; p++) e[p] = 0.0;
    static_for<C>([&](auto mm) KFVM_INLINE {
      constexpr int m = decltype(mm)::value, n = A > 0 ? PTab<D>::SL.slot[A > 0 ? A : 0][m] : m;
      constexpr int p = PTab<D>::PT.neg[n];
      if constexpr (!(p & zm)) e[p] = fma(w[z * C + m], t[n], e[p]);
    });
    static_for<D>([&](auto dd) KFVM_INLINE {
      static_for<ALL + 1>([&](auto pp) KFVM_INLINE {
        constexpr int d = decltype(dd)::value, p = decltype(pp)::value;
        if constexpr (!(zm >> d & 1) && !(p >> d & 1) && !(p & zm)) {
          const double ev = e[p], od = e[p | (1 << d)];
          e[p] = ev - od;
          e[p | (1 << d)] = ev + od;
        }
      });
    });
    static_for<ALL + 1>([&](auto ss) KFVM_INLINE {
      constexpr int s = decltype(ss)::value;
      if constexpr (!(s & zm)) out[parity_point(D, NQ, A, zm, s)] = e[s];
    });
  });
}

// Stencil values of a brick cell from one staged plane (corner: its box corner).
// The offset is opaque at each call: the planes do not change, so the compiler
// would otherwise keep one sweep's values for the next and spill them.
template <int D, class Bx>
__device__ __forceinline__ void load_stencil(const double *plane, int corner, double (&t)[SInfo<D>::C]) {
  asm volatile("" : "+v"(corner));
  const double *p = plane + corner;
  static_for<SInfo<D>::C>([&](auto nn) KFVM_INLINE {
    constexpr int n = decltype(nn)::value;
    constexpr int o = (StTab<D>::ST.off[n][0] + Bx::H) + Bx::LX * (StTab<D>::ST.off[n][1] + Bx::H) +
                      (D == 3 ? Bx::LX * Bx::LY * (StTab<D>::ST.off[n][2] + Bx::H) : 0);
    t[n] = p[o];
  });
}

// The brick at (i0,j0,k0) and its radius-2 halo, NV conserved planes, into LDS
// (box cells no stencil of a live cell reads are left as they are).
template <int D, int NV, class Bx>
__device__ __forceinline__ void stage_brick(const double *__restrict__ U, const Grid &g, int i0, int j0, int k0,
                                            int tid, double *lds) {
  constexpr int H = Bx::H, NP = Bx::N;
  const size_t nc = g.ncell;
  for (int idx = tid; idx < NP; idx += Bx::NT) {
    const int a = idx % Bx::LX, r = idx / Bx::LX, bb = r % Bx::LY, c = r / Bx::LY;
    const int ex = box_out<Bx::BX, H>(a), ey = box_out<Bx::BY, H>(bb);
    const int ez = D == 3 ? box_out<Bx::BZ, H>(c) : 0;
    const int gi = i0 + a - H, gj = j0 + bb - H, gk = D == 3 ? k0 + c - H : k0;
    const bool need = ex * ex + ey * ey + ez * ez <= H * H && gi < g.nx + H && gj < g.ny + H &&
                      (D == 2 || gk < g.nz + H);
    if (need) {
      const CellRef cr = map_cell<D, NV>(g, gi, gj, gk);
#pragma unroll
      for (int w = 0; w < NV; w++) lds[w * NP + idx] = ld(U, nc, cr, w);
    }
  }
}

// Wave-aggregated append of the marked cells to a list.
__device__ __forceinline__ void append_cells(bool mark, int cell, int *__restrict__ list, int *__restrict__ count) {
  const unsigned long long mask = __ballot(mark);
  if (mask) {
    const int lane = threadIdx.x & 63;
    const int leader = __ffsll((long long)mask) - 1;
    int base = 0;
    if (lane == leader) base = atomicAdd(count, __popcll(mask));
    base = __shfl(base, leader);
    if (mark) list[base + __popcll(mask & ((1ull << lane) - 1ull))] = cell;
  }
}

// Linear pass on a staged brick, one thread per cell, in the parity form: per
// variable one read of the stencil and one butterfly serve all face points, so
// the stencil crosses LDS once per variable.  Density and |m|^2 of the points
// stay in registers until the energy completes them (p/rho^gamma and the
// limiter's fast test); for the 54 points of the 3D 3x3 rule that takes one
// sweep over the variables per axis.
//   SURF   only the states on the brick's outer faces are stored, into the
//          surface planes SB from which the neighbouring bricks' k_flux_par
//          read them; otherwise every state goes to FS
//   LEARN  the learned WENO selection follows on the same brick (learned_tail)
template <int D, int NQ, bool SURF, bool LEARN>
__global__ __launch_bounds__(RBox<D>::NT, D == 3 && NQ == 3 ? 2 : 3) void k_linear_par(
    const double *__restrict__ U, double *__restrict__ FS, double *__restrict__ WI,
    double *__restrict__ thetaNew, const double *__restrict__ props, Grid g, const double *__restrict__ PW,
    int *__restrict__ ppList, int *__restrict__ ppCount, double *__restrict__ SB, Surf sb, LearnArgs la) {
  using Bx = RBox<D>;
  constexpr int C = SInfo<D>::C, Q = Shape<D, NQ>::Q, FQ = 2 * D * Q, H = Bx::H, NP = Bx::N;
  constexpr int AXG = D == 3 ? 1 : D;  // axes per sweep over the variables
  __shared__ double lds[5 * NP];
  const int nbx = (g.nx + Bx::BX - 1) / Bx::BX, nby = (g.ny + Bx::BY - 1) / Bx::BY;
  const int b = xcd_block(blockIdx.x, gridDim.x);
  const int i0 = (b % nbx) * Bx::BX, j0 = ((b / nbx) % nby) * Bx::BY, k0 = (b / (nbx * nby)) * Bx::BZ;
  const int tid = threadIdx.x;
  stage_brick<D, 5, Bx>(U, g, i0, j0, k0, tid, lds);
  __syncthreads();
  const int tx = tid % Bx::BX, ty = (tid / Bx::BX) % Bx::BY, tz = tid / (Bx::BX * Bx::BY);
  const int i = i0 + tx, j = j0 + ty, k = k0 + tz;
  if (i < g.nx && j < g.ny && (D == 2 || k < g.nz)) {  // no barrier inside
    const int cell = (k * g.ny + j) * g.nx + i;
    const int corner = (tz * Bx::LY + ty) * Bx::LX + tx;  // stencil box corner (-H,-H,-H)
    const int c0 = corner + H + Bx::LX * H + (D == 3 ? Bx::LX * Bx::LY * H : 0);
    double ref[5];
#pragma unroll
    for (int w = 0; w < 5; w++) ref[w] = lds[w * NP + c0];
    const PPBounds pb = pp_bounds_lds<D>(lds, c0, props, g, i, j, k, ref);
    const double gm1 = g.gamma - 1.0;
    // Fast test of the limiter: every density strictly inside the bounds and
    // every internal energy above its bound by more than rounding, without the
    // exact sequence's divisions.  A cell that fails, or only touches a bound,
    // goes to the exact sequence, which then decides.  The tests are formed where
    // their values are (keep_here): as a chain of conditions they were put off to
    // the end, with the values (3x3 rule: 256 registers and scratch, now 200;
    // 75 x 62 x 81 0.395 -> 0.367 ms, 2D 1024^2 0.099 -> 0.090).
    int bad = 0;
    static_for<D / AXG>([&](auto grp) KFVM_INLINE {
      constexpr int A0 = decltype(grp)::value * AXG;
      double rho[AXG * 2 * Q], msq[AXG * 2 * Q];
      static_for<5>([&](auto vv) KFVM_INLINE {
        constexpr int v = decltype(vv)::value;
        double t[C];
        load_stencil<D, Bx>(lds + v * NP, corner, t);
        parity_transform<D>(t);
        // opaque per variable, so that the coefficients stay scalar loads next
        // to their products instead of being hoisted out of the loop
        const double *w0 = PW;
        asm volatile("" : "+s"(w0));
        static_for<AXG>([&](auto ax) KFVM_INLINE {
          constexpr int A = A0 + decltype(ax)::value, P0 = (A - A0) * 2 * Q;
          double out[2 * Q];
          parity_points<D, NQ, A>(t, (const cdouble *)w0, out);
          __builtin_amdgcn_sched_barrier(0);
          if constexpr (SURF) {
            const int tA = A == 0 ? tx : (A == 1 ? ty : tz);
            const int last = A == 0 ? min(Bx::BX, g.nx - i0) - 1
                                    : (A == 1 ? min(Bx::BY, g.ny - j0) - 1 : min(Bx::BZ, g.nz - k0) - 1);
            const size_t T = size_t(sb.T[A]);
#pragma unroll
            for (int hi = 0; hi < 2; hi++)
              if (tA == (hi ? last : 0)) {
                double *d = SB + surf_index<D, Q>(sb, g, 2 * A + hi, i, j, k, 0, 0) + size_t(v) * T;
#pragma unroll
                for (int q = 0; q < Q; q++) d[size_t(q * 5) * T] = out[hi * Q + q];
              }
          } else {
            double *d = FS + fs_base(cell, FQ * 5) + size_t(A * 2 * Q * 5 + v) * FSB;
#pragma unroll
            for (int p = 0; p < 2 * Q; p++) d[size_t(p * 5) * FSB] = out[p];
          }
          if constexpr (v == 0) {
#pragma unroll
            for (int p = 0; p < 2 * Q; p++) {
              rho[P0 + p] = out[p];
              bad |= !((out[p] > pb.minDens) & (out[p] < pb.maxDens) & (out[p] > 0.0));
              keep_here(bad);
            }
          } else if constexpr (v < 4) {
#pragma unroll
            for (int p = 0; p < 2 * Q; p++) {
              msq[P0 + p] = v == 1 ? out[p] * out[p] : msq[P0 + p] + out[p] * out[p];
              keep_here(msq[P0 + p]);
            }
          } else {
#pragma unroll
            for (int p = 0; p < 2 * Q; p++) {
              const double lhs = (out[p] - 1e-14 * fabs(out[p]) - pb.minEint) * rho[P0 + p];
              bad |= !(lhs > 0.5 * msq[P0 + p]);
              keep_here(bad);
              if constexpr (!LEARN) msq[P0 + p] = out[p] - div_n(0.5 * msq[P0 + p], rho[P0 + p]);  // eint
            }
          }
        });
      });
      if constexpr (!LEARN) {
        // the KXRCF indicator's input p / rho^gamma, IT points per trip (one
        // pow's temporaries at a time, the points shifted down in registers)
        constexpr int NPT = AXG * 2 * Q, IT = NPT % 8 == 0 ? 8 : (NPT % 6 == 0 ? 6 : NPT);
        double *wi = WI + fs_base(cell, FQ) + size_t(A0 * 2 * Q) * FSB;
#pragma unroll 1
        for (int p0 = 0; p0 < NPT; p0 += IT) {
#pragma unroll
          for (int p = 0; p < IT; p++) {
            wi[size_t(p0 + p) * FSB] = (gm1 * msq[p]) * pow_pos(rho[p], -g.gamma);
            __builtin_amdgcn_sched_barrier(0);
          }
#pragma unroll
          for (int p = 0; p + IT < NPT; p++) {
            rho[p] = rho[p + IT];
            msq[p] = msq[p + IT];
          }
        }
      }
    });
    // Cells whose states violate a bound go to a list for the limiter's exact
    // sequence (keeping it out of this kernel keeps its waves convergent).
    if (!bad) thetaNew[cell] = 1.0;
    append_cells(bad != 0, cell, ppList, ppCount);
  }
  // every thread of the block, live or not, runs the selection (barriers, MFMA)
  if (LEARN) learned_tail<D>(lds, la, g, i0, j0, k0, tid);
}

// Rows of the listed cells: row t holds the F*Q*5 face states of one cell,
// value (f*Q + q)*5 + v.
template <int D, int NQ>
struct RowShape {
  static constexpr int Q = Shape<D, NQ>::Q, F = Shape<D, NQ>::F, N = F * Q * 5;
};

// One group of LPG lanes per listed cell (lane pl = face point pl): the
// point's five linear values from the stencil gathered through the boundary
// index map, in the parity form of the other kernels (every lane transforms
// the cell's stencil, forms its own axis' points and keeps its own), the
// limiter with group reductions, the limited states into row rowBase + (an
// atomic count), and pos[c] = row.
template <int D, int NQ>
__global__ __launch_bounds__(BLK) void k_pp_rows(const double *__restrict__ U, double *__restrict__ rows,
                                                 int *__restrict__ pos, double *__restrict__ thetaNew,
                                                 const double *__restrict__ props,
                                                 const double *__restrict__ wflag, Grid g,
                                                 const double *__restrict__ PW, const int *__restrict__ list,
                                                 const int *__restrict__ count, const int *__restrict__ wenoCount,
                                                 int *__restrict__ rowCount) {
  constexpr int C = SInfo<D>::C, Q = Shape<D, NQ>::Q, FQ = Shape<D, NQ>::F * Q, LPG = PPGroup<FQ>::LPG;
  constexpr int GPW = 64 / LPG;
  const int n = *count;
  const int lane = threadIdx.x & 63, pl = lane % LPG;
  const int gid = (blockIdx.x * (BLK / 64) + (threadIdx.x >> 6)) * GPW + lane / LPG;
  const int ngroups = gridDim.x * (BLK / 64) * GPW;
  const size_t nc = g.ncell;
  const int rowBase = *wenoCount;  // the WENO cells' rows come first
  for (int t = gid; t < n; t += ngroups) {
    const int c = list[t];
    if (wflag[c] != 0.0) continue;  // uniform over the group
    int i, j, k;
    cell_ijk<D>(c, g, i, j, k);
    double ref[5];
#pragma unroll
    for (int w = 0; w < 5; w++) ref[w] = U[size_t(w) * nc + c];
    const PPBounds pb = grp_pp_bounds<D, LPG>(U, props, g, i, j, k, ref, pl);
    const bool own = pl < FQ;
    double st[5];
#pragma unroll 1
    for (int v = 0; v < 5; v++) {
      double s[C];
      static_for<C>([&](auto mm) KFVM_INLINE {
        constexpr int m = decltype(mm)::value;
        constexpr int ox = StTab<D>::ST.off[m][0], oy = StTab<D>::ST.off[m][1], oz = StTab<D>::ST.off[m][2];
        s[m] = load_u<D, 5>(U, g, i + ox, j + oy, k + oz, v);
      });
      parity_transform<D>(s);
      double mine = ref[0];
      const double *w0 = PW;
      asm volatile("" : "+s"(w0));
      static_for<D>([&](auto ax) KFVM_INLINE {
        constexpr int A = decltype(ax)::value;
        double out[2 * Q];
        parity_points<D, NQ, A>(s, (const cdouble *)w0, out);
#pragma unroll
        for (int p = 0; p < 2 * Q; p++) mine = pl == A * 2 * Q + p ? out[p] : mine;
      });
#pragma unroll
      for (int w = 0; w < 5; w++) st[w] = w == v ? (own ? mine : ref[w]) : (v == 0 ? 0.0 : st[w]);
    }
    const double thD = grp_min<LPG>(own ? dens_theta(1.0, st[0], pb) : 1.0);
    const bool mixD = thD > 0.0 && thD < 1.0, repD = !mixD && thD < 1.0;
#pragma unroll
    for (int w = 0; w < 5; w++) st[w] = repD ? ref[w] : (mixD ? ref[w] + thD * (st[w] - ref[w]) : st[w]);
    double thE = 1.0;
    if (own && !(Hydro::eint(st) > pb.minEint)) thE = eint_pos(pb.minEint, ref, st);
    const double thP = grp_min<LPG>(thE);
    const bool mixP = thP > 0.0 && thP < 1.0, repP = !mixP && thP < 1.0;
#pragma unroll
    for (int w = 0; w < 5; w++) st[w] = repP ? ref[w] : (mixP ? ref[w] + thP * (st[w] - ref[w]) : st[w]);
    int row = 0;
    if (pl == 0) row = rowBase + atomicAdd(rowCount, 1);
    row = __shfl(row, lane - pl);
    if (own) {
      double *dst = rows + size_t(row) * (FQ * 5) + pl * 5;
#pragma unroll
      for (int w = 0; w < 5; w++) dst[w] = st[w];
    }
    if (pl == 0) {
      thetaNew[c] = fmin(thD, thP);
      pos[c] = row;
    }
  }
}

// --------------------------------------------------------- k_flux_par
template <int D, int NQ>
struct FluxPar {
  using Bx = RBox<D>;
  static constexpr int Q = Shape<D, NQ>::Q;
  // upper outer faces of the brick, x, y (and z): one per transverse cell
  static constexpr int EX = Bx::BY * Bx::BZ, EY = Bx::BX * Bx::BZ, EZ = D == 3 ? Bx::BX * Bx::BY : 0;
  static constexpr int NE = EX + EY + EZ;
  static constexpr int RX = Bx::BX + 2, RY = Bx::BY + 2, RZ = D == 3 ? Bx::BZ + 2 : 1;
  // LDS: the staged brick, later the last axis' upper states and face fluxes
  static constexpr int XS = Bx::NT * Q * 5, XCH = XS + Bx::NT * 5;
  static constexpr int LDS = 5 * Bx::N > XCH ? 5 * Bx::N : XCH;
  static constexpr int UN = Q == 4 ? 2 : Q;  // face points solved per trip of the point loop
};

// Move a double by DPP within rows of 16 lanes (0x111: from lane - 1, 0x101:
// from lane + 1); the lanes without a source keep their own value.
template <int CTRL>
__device__ __forceinline__ double dpp_move(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = int(b), hi = int(b >> 32);
  const int l2 = __builtin_amdgcn_update_dpp(lo, lo, CTRL, 0xf, 0xf, false);
  const int h2 = __builtin_amdgcn_update_dpp(hi, hi, CTRL, 0xf, 0xf, false);
  return __longlong_as_double((long long)(((unsigned long long)(unsigned)h2 << 32) | (unsigned)l2));
}

// One thread per cell of a 16 x 4 x 4 (2D: 16 x 16) brick.  Axis by axis a
// thread forms the states of its cell at the 2 Q points of the axis' two faces
// from the staged brick (the parity form: 33 products for the 8 points of a
// variable in 3D), takes the lower neighbour's upper states (adjacent lanes in
// x, 16 lanes away in y of a 3D brick, through LDS along the last axis, where
// the brick's planes are no longer needed) and solves its lower face at every
// point, keeping the flux integrated over the face in five registers.  The
// brick's upper outer faces are (face, point) work items spread over all
// threads.  States beyond the brick come from the surface planes of the
// linear pass or from rows; a face shared by two bricks is solved in both from
// the same two states.  The variables are held rotated, the axis' normal
// momentum first, so that one solver serves every axis.
template <int D, int NQ, bool HLLC>
__global__ __launch_bounds__(RBox<D>::NT, 2) void k_flux_par(const double *__restrict__ U,
                                                             const double *__restrict__ PW,
                                                             const double *__restrict__ rows,
                                                             const int *__restrict__ pos,
                                                             const double *__restrict__ SB, Surf sb, Grid g,
                                                             RKArgs a) {
  using Bx = RBox<D>;
  using FP = FluxPar<D, NQ>;
  constexpr int C = SInfo<D>::C, Q = FP::Q, NP = Bx::N, NT = Bx::NT, RN = RowShape<D, NQ>::N;
  constexpr int BX = Bx::BX, BY = Bx::BY, BZ = Bx::BZ;
  static_assert(BX == 16 && NT == BLK, "DPP rows of 16 cells, one brick per block of BLK threads");
  static_assert(Q % FP::UN == 0, "whole trips of the point loop");
  __shared__ double lds[FP::LDS];
  __shared__ double xt[FP::NE * Q * 5];
  __shared__ int rowTab[FP::RX * FP::RY * FP::RZ];

  const int nbx = (g.nx + BX - 1) / BX, nby = (g.ny + BY - 1) / BY;
  const int b = xcd_block(blockIdx.x, gridDim.x);
  const int i0 = (b % nbx) * BX, j0 = ((b / nbx) % nby) * BY, k0 = (b / (nbx * nby)) * BZ;
  const int tid = threadIdx.x;
  const size_t nc = g.ncell;
  stage_brick<D, 5, Bx>(U, g, i0, j0, k0, tid, lds);
  // rows of the brick's cells and their face neighbours (-1: no row; cells
  // beyond a wall are never read, periodic ones wrap)
  for (int e = tid; e < FP::RX * FP::RY * FP::RZ; e += NT) {
    const int x = i0 - 1 + e % FP::RX, y = j0 - 1 + (e / FP::RX) % FP::RY;
    const int z = D == 3 ? k0 - 1 + e / (FP::RX * FP::RY) : k0;
    const bool wall = (x < 0 && g.bc[0] != 0) || (x >= g.nx && g.bc[1] != 0) || (y < 0 && g.bc[2] != 0) ||
                      (y >= g.ny && g.bc[3] != 0) ||
                      (D == 3 && ((z < 0 && g.bc[4] != 0) || (z >= g.nz && g.bc[5] != 0)));
    int r = -1;
    if (!wall) {
      const int xw = x < 0 ? x + g.nx : (x >= g.nx ? x - g.nx : x);
      const int yw = y < 0 ? y + g.ny : (y >= g.ny ? y - g.ny : y);
      const int zw = D == 3 ? (z < 0 ? z + g.nz : (z >= g.nz ? z - g.nz : z)) : z;
      if (xw >= 0 && xw < g.nx && yw >= 0 && yw < g.ny && zw >= 0 && (D == 2 || zw < g.nz))
        r = pos[(size_t(zw) * g.ny + yw) * g.nx + xw];
    }
    rowTab[e] = r;
  }
  __syncthreads();

  const int tx = tid % BX, ty = (tid / BX) % BY, tz = tid / (BX * BY);
  const int lastX = min(BX, g.nx - i0) - 1, lastY = min(BY, g.ny - j0) - 1;
  const int lastZ = D == 3 ? min(BZ, g.nz - k0) - 1 : 0;
  const bool live = tx <= lastX && ty <= lastY && tz <= lastZ;
  const size_t c = live ? (size_t(k0 + tz) * g.ny + (j0 + ty)) * g.nx + i0 + tx : 0;
  const int corner = (tz * Bx::LY + ty) * Bx::LX + tx;
  auto row_at = [&](int x, int y, int z) {  // brick-local coordinates, -1 .. B
    return rowTab[(x + 1) + FP::RX * ((y + 1) + FP::RY * (D == 3 ? z + 1 : 0))];
  };
  const int myRow = live ? row_at(tx, ty, tz) : -1;
  double vmax = 0.0;

  // Source of the states on face fn of the cell at brick-local (x,y,z) just
  // outside the brick along axis ax: value (q, v) at p[q * qs + v * vs], or
  // p = nullptr at a wall (the mirror of the inner state).
  struct Outer {
    const double *p;
    size_t qs, vs;
  };
  auto outer = [&](int ax, int fn, int x, int y, int z) {
    Outer o{nullptr, 0, 0};
    int gx = i0 + x, gy = j0 + y, gz = k0 + z;
    const int n_ax = ax == 0 ? g.nx : (ax == 1 ? g.ny : g.nz);
    const int co = ax == 0 ? gx : (ax == 1 ? gy : gz);
    if (co < 0 || co >= n_ax) {
      const int bLo = ax == 0 ? g.bc[0] : (ax == 1 ? g.bc[2] : g.bc[4]);
      const int bHi = ax == 0 ? g.bc[1] : (ax == 1 ? g.bc[3] : g.bc[5]);
      if ((co < 0 ? bLo : bHi) != 0) return o;
      const int w = co < 0 ? co + n_ax : co - n_ax;
      if (ax == 0) gx = w;
      else if (ax == 1) gy = w;
      else gz = w;
    }
    const int r = row_at(x, y, z);
    if (r >= 0) {
      o.p = rows + size_t(r) * RN + fn * Q * 5;
      o.qs = 5;
      o.vs = 1;
    } else {
      const size_t T = size_t(ax == 0 ? sb.T[0] : (ax == 1 ? sb.T[1] : sb.T[2]));
      const int hi = fn & 1, cc = ax == 0 ? gx : (ax == 1 ? gy : gz);
      const int t = ax == 0 ? gz * g.ny + gy : (ax == 1 ? gz * g.nx + gx : gy * g.nx + gx);
      const int pl = cc / (ax == 0 ? BX : (ax == 1 ? BY : BZ)) + hi;
      const size_t off = size_t(ax == 0 ? sb.off[0] : (ax == 1 ? sb.off[1] : sb.off[2]));
      o.p = SB + off + (size_t(pl * 2 + (hi ? 0 : 1)) * (Q * 5)) * T + t;
      o.qs = 5 * T;
      o.vs = T;
    }
    return o;
  };
  auto solve = [&](const double *uL, const double *uR, double *F) {
    if constexpr (HLLC) return Hydro::solve_hllc<0>(g.gamma, uL, uR, F);
    else return Hydro::solve_hll<0>(g.gamma, g.rs == 0, uL, uR, F);
  };

  // lower-face fluxes of this cell, integrated over the face, rotated
  double S[D][5];
  static_for<D>([&](auto ax) KFVM_INLINE {
    constexpr int A = decltype(ax)::value;
    constexpr bool LAST = A == D - 1;
    constexpr int rv[5] = {0, 1 + A, 1 + (A + 1) % 3, 1 + (A + 2) % 3, 4};
    const int tA = A == 0 ? tx : (A == 1 ? ty : tz);
    const int lastA = A == 0 ? lastX : (A == 1 ? lastY : lastZ);
    double pt[5][2 * Q];
    {
      const double *w0 = PW;
      asm volatile("" : "+s"(w0));
#pragma unroll
      for (int w = 0; w < 5; w++) {
        double t[C];
        load_stencil<D, Bx>(lds + rv[w] * NP, corner, t);
        parity_transform<D>(t);
        parity_points<D, NQ, A>(t, (const cdouble *)w0, pt[w]);
        __builtin_amdgcn_sched_barrier(0);  // one variable's stencil in registers at a time
      }
    }
    if (myRow >= 0) {
      const double *r = rows + size_t(myRow) * RN + 2 * A * Q * 5;
#pragma unroll
      for (int p = 0; p < 2 * Q; p++)
#pragma unroll
        for (int w = 0; w < 5; w++) pt[w][p] = r[p * 5 + rv[w]];
    }
    if (LAST) {
      __syncthreads();  // every thread has read its stencils: the planes are free
#pragma unroll
      for (int q = 0; q < Q; q++)
#pragma unroll
        for (int w = 0; w < 5; w++) lds[(q * 5 + w) * NT + tid] = pt[w][Q + q];
    }
    if (live && tA == lastA) {
      const int e = A == 0 ? ty + BY * tz : (A == 1 ? FP::EX + tx + BX * tz : FP::EX + FP::EY + tx + BX * ty);
#pragma unroll
      for (int q = 0; q < Q; q++)
#pragma unroll
        for (int w = 0; w < 5; w++) xt[(e * Q + q) * 5 + w] = pt[w][Q + q];
    }
    // the lower neighbour's upper states
    double nb[5][Q];
    if (LAST) __syncthreads();
#pragma unroll
    for (int q = 0; q < Q; q++)
#pragma unroll
      for (int w = 0; w < 5; w++) {
        if (LAST) nb[w][q] = lds[(q * 5 + w) * NT + (tA > 0 ? tid - (A == 1 ? BX : BX * BY) : tid)];
        else if (A == 0) nb[w][q] = dpp_move<0x111>(pt[w][Q + q]);
        else nb[w][q] = __shfl_up(pt[w][Q + q], 16);
      }
    if (live && tA == 0) {
      const Outer o = outer(A, 2 * A + 1, A == 0 ? -1 : tx, A == 1 ? -1 : ty, A == 2 ? -1 : tz);
      const unsigned m = g.negmask[2 * A];
#pragma unroll
      for (int q = 0; q < Q; q++)
#pragma unroll
        for (int w = 0; w < 5; w++)
          nb[w][q] = o.p ? o.p[q * o.qs + rv[w] * o.vs] : (((m >> rv[w]) & 1u) ? -pt[w][q] : pt[w][q]);
    }
#pragma unroll
    for (int w = 0; w < 5; w++) S[A][w] = 0.0;
#pragma unroll 1
    for (int q0 = 0; q0 < Q; q0 += FP::UN) {
#pragma unroll
      for (int u = 0; u < FP::UN; u++) {
        double uL[5], uR[5], Fl[5];
#pragma unroll
        for (int w = 0; w < 5; w++) {
          uL[w] = nb[w][u];
          uR[w] = pt[w][u];
        }
        const double sp = solve(uL, uR, Fl);
        if (live) vmax = sp > vmax ? sp : vmax;
        const double wq = face_weight<D, NQ>(g, q0 + u);
#pragma unroll
        for (int w = 0; w < 5; w++) S[A][w] += wq * Fl[w];
        __builtin_amdgcn_sched_barrier(0);  // one solve's temporaries at a time
      }
#pragma unroll
      for (int q = 0; q + FP::UN < Q; q++)
#pragma unroll
        for (int w = 0; w < 5; w++) {
          nb[w][q] = nb[w][q + FP::UN];
          pt[w][q] = pt[w][q + FP::UN];
        }
    }
    if (LAST) {
#pragma unroll
      for (int w = 0; w < 5; w++) lds[FP::XS + w * NT + tid] = S[A][w];
    }
  });

  // upper outer faces: one (face, point) per work item, in place over the
  // inner cell's states
#pragma unroll 1
  for (int it = tid; it < FP::NE * Q; it += NT) {
    const int f = it / Q, q = it % Q;
    const int ax = f < FP::EX ? 0 : (f < FP::EX + FP::EY ? 1 : 2);
    int x, y, z;
    if (ax == 0) {
      x = lastX;
      y = f % BY;
      z = f / BY;
    } else if (ax == 1) {
      x = (f - FP::EX) % BX;
      y = lastY;
      z = (f - FP::EX) / BX;
    } else {
      x = (f - FP::EX - FP::EY) % BX;
      y = (f - FP::EX - FP::EY) / BX;
      z = lastZ;
    }
    if (x > lastX || y > lastY || z > lastZ) continue;
    double uL[5], uR[5], Fl[5];
#pragma unroll
    for (int w = 0; w < 5; w++) uL[w] = xt[it * 5 + w];
    const Outer o = outer(ax, 2 * ax, x + (ax == 0), y + (ax == 1), z + (ax == 2));
    const unsigned m = ax == 0 ? g.negmask[1] : (ax == 1 ? g.negmask[3] : g.negmask[5]);
#pragma unroll
    for (int w = 0; w < 5; w++) {
      const int v = rotated_var<5>(w, ax);
      uR[w] = o.p ? o.p[q * o.qs + v * o.vs] : (((m >> v) & 1u) ? -uL[w] : uL[w]);
    }
    const double sp = solve(uL, uR, Fl);
    vmax = sp > vmax ? sp : vmax;
#pragma unroll
    for (int w = 0; w < 5; w++) xt[it * 5 + w] = Fl[w];
  }
  __syncthreads();

  // divergence: the upper neighbours' lower fluxes, or the outer faces'
  double rhs[5];
  const double rdx = 1.0 / g.dx, rdy = 1.0 / g.dy, rdz = 1.0 / g.dz;
  static_for<D>([&](auto ax) KFVM_INLINE {
    constexpr int A = decltype(ax)::value;
    constexpr bool LAST = A == D - 1;
    constexpr int rv[5] = {0, 1 + A, 1 + (A + 1) % 3, 1 + (A + 2) % 3, 4};
    const int tA = A == 0 ? tx : (A == 1 ? ty : tz);
    const int lastA = A == 0 ? lastX : (A == 1 ? lastY : lastZ);
    const double rd = A == 0 ? rdx : (A == 1 ? rdy : rdz);
    double up[5];
#pragma unroll
    for (int w = 0; w < 5; w++) {
      if (LAST) up[w] = lds[FP::XS + w * NT + (tA < lastA ? tid + (A == 1 ? BX : BX * BY) : tid)];
      else if (A == 0) up[w] = dpp_move<0x101>(S[A][w]);
      else up[w] = __shfl_down(S[A][w], 16);
    }
    if (live && tA == lastA) {
      const int e = A == 0 ? ty + BY * tz : (A == 1 ? FP::EX + tx + BX * tz : FP::EX + FP::EY + tx + BX * ty);
#pragma unroll
      for (int w = 0; w < 5; w++) up[w] = 0.0;
#pragma unroll
      for (int q = 0; q < Q; q++) {
        const double wq = face_weight<D, NQ>(g, q);
#pragma unroll
        for (int w = 0; w < 5; w++) up[w] += wq * xt[(e * Q + q) * 5 + w];
      }
    }
#pragma unroll
    for (int w = 0; w < 5; w++) {
      const double d = (S[A][w] - up[w]) * rd;
      rhs[rv[w]] = A == 0 ? d : rhs[rv[w]] + d;
    }
  });

  // RK register update and error norm (the epilogue of k_flux_rk); 2D batches:
  // the brick's slice and its step size
  const int slice = D == 2 ? k0 : 0;
  const double betaDt = a.sliceDt ? a.beta * a.sliceDt[slice] : a.betaDt;
  const double bhatDt = a.sliceDt ? a.bhat * a.sliceDt[slice] : a.bhatDt;
  double errLoc = 0.0, posLoc = 1.0;
  const bool write = !a.sliceWrite || a.sliceWrite[slice] != 0;
  if (live) rk_epilogue<5>(a, U, c, nc, rhs, betaDt, bhatDt, write, errLoc, posLoc);
  __syncthreads();  // lds is free again
  const double bmax = block_max(vmax, lds, tid);
  if (tid == 0 && bmax > 0.0) atomicMax(a.vmaxBits + slice, (unsigned long long)__double_as_longlong(bmax));
  if (a.mode == RK_FSAL) {
    const double es = block_sum(errLoc, lds, tid);
    const double pm = block_min(posLoc, lds, tid);
    if (tid == 0) {
      a.errPartial[b] = es;
      a.posPartial[b] = pm;
    }
  }
}

}  // namespace dev
}  // namespace kfvm
