// The GLM-MHD linear pass in the mirror-symmetric form of parity5.hpp.
//
//   k_mhd_linear_par  KernelLinearRecon_K incl. the source branch
//                     (Stencil_K.H:32-118), the KXRCF input (Numeric_K.H:315-379),
//                     the limiter's fast test (Common_K.H:299-643) and the
//                     cleaning-speed maxima (SpeedEstimate_K, MHD_GLM_K.H:213-310)
#pragma once

namespace kfvm {
namespace dev {

// One thread per cell of the 16 x 8 x 4 brick that k_mhd_linear stages (nine
// variables and their radius-2 halo, 138 KB: one workgroup of 8 waves per CU).
// Per face axis one sweep over the variables (and one for the interior
// points): a variable's stencil is read and transformed once for all points of
// the sweep, its values stored, and only the sums a point's later tests need
// stay in registers (density, |m|^2, |B|^2, the energy as it loses its kinetic,
// magnetic and cleaning parts).  32 points of 33 products each take 4 x (33 +
// 24) operations after the 60 of the butterfly instead of 1056, which leaves
// the pass to the 2.3 KB it stores per cell.
// IND: the KXRCF indicator's input is written (not for the learned selection).
template <int D, int NQ, bool IND>
__global__ __launch_bounds__(MBox<D>::NT, 2) void k_mhd_linear_par(
    const double *__restrict__ U, double *__restrict__ FS, double *__restrict__ SRC, double *__restrict__ WI,
    double *__restrict__ thetaNew, double *__restrict__ spd, const double *__restrict__ props, Grid g,
    const double *__restrict__ PW, int *__restrict__ ppList, int *__restrict__ ppCount) {
  using Bx = MBox<D>;
  constexpr int C = SInfo<D>::C, H = Bx::H, NP = Bx::N;
  constexpr int FQ = MShape<D, NQ>::FQ;
  __shared__ double lds[9 * NP];
  const int nbx = (g.nx + Bx::BX - 1) / Bx::BX, nby = (g.ny + Bx::BY - 1) / Bx::BY;
  const int b = xcd_block(blockIdx.x, gridDim.x);
  const int i0 = (b % nbx) * Bx::BX, j0 = ((b / nbx) % nby) * Bx::BY, k0 = (b / (nbx * nby)) * Bx::BZ;
  const int tid = threadIdx.x;
  const size_t nc = g.ncell;
  stage_brick<D, 9, Bx>(U, g, i0, j0, k0, tid, lds);
  __syncthreads();
  const int tx = tid % Bx::BX, ty = (tid / Bx::BX) % Bx::BY, tz = tid / (Bx::BX * Bx::BY);
  const int i = i0 + tx, j = j0 + ty, k = k0 + tz;
  if (i >= g.nx || j >= g.ny || (D == 3 && k >= g.nz)) return;  // no barrier follows
  const int cell = (k * g.ny + j) * g.nx + i;
  const int corner = (tz * Bx::LY + ty) * Bx::LX + tx;  // stencil box corner (-H,-H,-H)
  const int c0 = corner + H + Bx::LX * H + (D == 3 ? Bx::LX * Bx::LY * H : 0);
  double ref[9];
#pragma unroll
  for (int w = 0; w < 9; w++) ref[w] = lds[w * NP + c0];
  const PPBounds pb = pp_bounds_lds<D, Bx>(lds, c0, props, g, i, j, k, ref);
  const double gm1 = g.gamma - 1.0;
  double maxLam = 0.0, maxVel = 0.0;
  int bad = 0;
  // axes 0 .. D - 1: the faces; D: the interior points
  static_for<D + 1>([&](auto ss) KFVM_INLINE {
    constexpr bool FACE = decltype(ss)::value < D;
    constexpr int A = FACE ? decltype(ss)::value : -1, N = ParPts<D, NQ, A>::N;
    double m1[FACE ? N : 1], msq[N], bx[FACE ? N : 1], bsq[N], e[N];
    double eMax = 0.0;  // largest energy of the points: its rounding is the test's margin
    static_for<9>([&](auto oo) KFVM_INLINE {
      // momenta, field, cleaning variable, energy; the density last, which
      // completes the points
      constexpr int o = decltype(oo)::value, v = o < 3 ? o + 1 : (o < 7 ? o + 2 : (o == 7 ? 4 : 0));
      double out[N];
      {
        double t[C];
        load_stencil<D, Bx>(lds + v * NP, corner, t);
        parity_transform<D>(t);
        const double *w0 = PW + (FACE ? 0 : parity_face_types(D, NQ) * C);
        asm volatile("" : "+s"(w0));
        parity_points<D, NQ, A>(t, (const cdouble *)w0, out);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (FACE) {
        double *d = FS + fs_base(cell, FQ * 9) + size_t(A * N * 9 + v) * FSB;
#pragma unroll
        for (int p = 0; p < N; p++) d[size_t(p * 9) * FSB] = out[p];
      } else {
#pragma unroll
        for (int p = 0; p < N; p++) SRC[(size_t(p) * 9 + v) * nc + cell] = out[p];
      }
#pragma unroll
      for (int p = 0; p < N; p++) {
        const double x = out[p];
        if constexpr (v >= 1 && v <= 3) {
          if constexpr (v == 1 && FACE) m1[p] = x;
          msq[p] = v == 1 ? x * x : msq[p] + x * x;
          keep_here(msq[p]);
        } else if constexpr (v >= 5 && v <= 7) {
          if constexpr (v == 5 && FACE) bx[p] = x;
          bsq[p] = v == 5 ? x * x : bsq[p] + x * x;
          keep_here(bsq[p]);
        } else if constexpr (v == 8) {
          e[p] = -0.5 * x * x;
          keep_here(e[p]);
        } else if constexpr (v == 4) {
          e[p] = x - 0.5 * bsq[p] + e[p];
          eMax = fmax(eMax, fabs(x));
          keep_here(e[p]);
          keep_here(eMax);
        } else {
          const double ir = rcp_n(x), ei = e[p] - 0.5 * msq[p] * ir;
          // beyond the bound by more than rounding (see k_linear_par)
          bad |= !((x > pb.minDens) & (x < pb.maxDens) & (x > 0.0) & (ei - 1e-14 * eMax > pb.minEint));
          keep_here(bad);
          if constexpr (FACE) {
            // fastest magnetosonic speed + |u| and |u|, x-components on every face
            const double vel = fabs(m1[p] * ir);
            const double asq = g.gamma * (gm1 * ei) * ir, absq = asq + bsq[p] * ir, blsq = bx[p] * bx[p] * ir;
            const double lam = sqrt_n(0.5 * (absq + sqrt_n(fmax(absq * absq - 4.0 * asq * blsq, 0.0)))) + vel;
            maxVel = vel > maxVel ? vel : maxVel;
            maxLam = lam > maxLam ? lam : maxLam;
            keep_here(maxVel);
            keep_here(maxLam);
            if constexpr (IND) {
              double wi = (gm1 * ei) * pow_pos(x, -g.gamma);
              keep_here(wi);
              WI[fs_base(cell, FQ) + size_t(A * N + p) * FSB] = wi;
            }
            __builtin_amdgcn_sched_barrier(0);
          }
        }
      }
      __builtin_amdgcn_sched_barrier(0);
    });
  });
  spd[cell] = maxLam;
  spd[nc + cell] = maxVel;
  if (!bad) thetaNew[cell] = 1.0;
  append_cells(bad != 0, cell, ppList, ppCount);
}

}  // namespace dev
}  // namespace kfvm
