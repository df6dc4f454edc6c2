// Euler flux kernel of the 3D runs with the learned selection: the divergence
// summed face point by face point.
//
// The trained 3D network scales the pressure deviations of a stencil by their
// largest, so where the pressure is constant (along a contact) it reads the
// rounding of the state, and which cells it picks changes with every change in
// the order of any sum: 1e-6 in the density of the 256^3 planar Riemann run
// within one step, where every other configuration agrees to 1e-15.  3D Euler
// runs with the network therefore keep the order of operations its results were
// taken with: dense linear products (k_linear_fused), this kernel and
// Hydro::solve_hllc_pt, and so do evaluations with WENO on every cell, which a
// run whose network picks every cell equals bit for bit.  All other runs use
// k_flux_rk / k_flux_par.
//
//   k_flux_points  Common_K.H:180-297, Numeric_K.H:109-290
#pragma once

namespace kfvm {
namespace dev {

template <int DIR>
__device__ inline double riemann_points(const Grid &g, const double *uL, const double *uR, double *Fl) {
  if (g.rs == 2) return Hydro::solve_hllc_pt<DIR>(g.gamma, uL, uR, Fl);
  return Hydro::solve_hll<DIR>(g.gamma, g.rs == 0, uL, uR, Fl);
}

template <int NQ>
__global__ __launch_bounds__(BLK) void k_flux_points(const double *__restrict__ U,
                                                     const double *__restrict__ FS, Grid g, RKArgs a) {
  constexpr int D = 3, NV = 5;
  using Bk = Brick<D>;
  constexpr int Q = Shape<D, NQ>::Q;
  __shared__ double fl[NV][Bk::NF];
  // compact WENO rows of the brick's cells and their face neighbours (Euler
  // sparse WENO; -1: states in FS)
  constexpr int RX = Bk::X + 2, RY = Bk::Y + 2, RZ = D == 3 ? Bk::Z + 2 : 1;
  __shared__ int rowTab[RX * RY * RZ];
  __shared__ double sh[BLK];
  const int tid = threadIdx.x + Bk::X * (threadIdx.y + Bk::Y * threadIdx.z);
  // one-dimensional grid of bricks, x fastest, renumbered per XCD
  const int nbx = (g.nx + Bk::X - 1) / Bk::X, nby = (g.ny + Bk::Y - 1) / Bk::Y;
  const int b = xcd_block(blockIdx.x, gridDim.x);
  const int bzi = b / (nbx * nby);
  const int i0 = (b % nbx) * Bk::X, j0 = ((b / nbx) % nby) * Bk::Y, k0 = bzi * Bk::Z;
  const int ci = i0 + threadIdx.x, cj = j0 + threadIdx.y, ck = k0 + threadIdx.z;
  const bool live = ci < g.nx && cj < g.ny && (D == 2 || ck < g.nz);
  const size_t nc = g.ncell;
  const size_t c = live ? (size_t(ck) * g.ny + cj) * g.nx + ci : 0;
  double vmax = 0.0, errLoc = 0.0, posLoc = 1.0;
  // 2D batches: the brick's slice (blockIdx.z) and its step size
  const int slice = D == 2 ? bzi : 0;
  const double betaDt = a.sliceDt ? a.beta * a.sliceDt[slice] : a.betaDt;
  const double bhatDt = a.sliceDt ? a.bhat * a.sliceDt[slice] : a.bhatDt;
  double rhs[NV];
#pragma unroll
  for (int v = 0; v < NV; v++) rhs[v] = 0.0;
  const double rdx = 1.0 / g.dx, rdy = 1.0 / g.dy, rdz = 1.0 / g.dz;

  const bool useRows = a.pos != nullptr;
  if (useRows) {
    for (int e = tid; e < RX * RY * RZ; e += BLK) {
      const int x = i0 - 1 + e % RX, y = j0 - 1 + (e / RX) % RY, z = D == 3 ? k0 - 1 + e / (RX * RY) : k0;
      // a cell beyond a non-periodic edge is never read (its face takes the
      // boundary state); a periodic one wraps
      const bool wall = (x < 0 && g.bc[0] != 0) || (x >= g.nx && g.bc[1] != 0) || (y < 0 && g.bc[2] != 0) ||
                        (y >= g.ny && g.bc[3] != 0) ||
                        (D == 3 && ((z < 0 && g.bc[4] != 0) || (z >= g.nz && g.bc[5] != 0)));
      int r = -1;
      if (!wall) {
        const int xw = x < 0 ? x + g.nx : (x >= g.nx ? x - g.nx : x);
        const int yw = y < 0 ? y + g.ny : (y >= g.ny ? y - g.ny : y);
        const int zw = D == 3 ? (z < 0 ? z + g.nz : (z >= g.nz ? z - g.nz : z)) : z;
        if (xw >= 0 && xw < g.nx && yw >= 0 && yw < g.ny && zw >= 0 && (D == 2 || zw < g.nz))
          r = a.pos[(size_t(zw) * g.ny + yw) * g.nx + xw];
      }
      rowTab[e] = r;
    }
    __syncthreads();
  }
  auto row_of = [&](int x, int y, int z) {
    if (!useRows) return -1;
    const int e = (x - i0 + 1) + RX * ((y - j0 + 1) + RY * (D == 3 ? z - k0 + 1 : 0));
    return rowTab[e];
  };

  // Face items (the same for every face point q): d0 = t | dir << 20 |
  // needed << 30 (-1: padding), and for each side the source of its states:
  // a cell index (>= 0, its FS slots), a compact WENO row r (-(r + 2)), or the
  // mirror of the other side (-1: a wall), resolved once per brick into LDS
  // (each thread reads back only the items it wrote).
  __shared__ int fd0[Bk::PF], fdL[Bk::PF], fdR[Bk::PF];
  constexpr int MIRROR = -1;
  auto describe = [&](int w, int &d0, int &sL, int &sR) {
    // padded work item w -> face t of the unpadded numbering (x, then y, then z faces)
    int dir, fi, fj, fk, t;
    bool pad = false;
    if (w < Bk::PXF) {
      pad = w >= Bk::NXF;
      t = w;
      dir = 0;
      fi = t % (Bk::X + 1);
      fj = (t / (Bk::X + 1)) % Bk::Y;
      fk = t / ((Bk::X + 1) * Bk::Y);
    } else if (w < Bk::PXF + Bk::PYF) {
      const int u = w - Bk::PXF;
      pad = u >= Bk::NYF;
      t = Bk::NXF + u;
      dir = 1;
      fi = u % Bk::X;
      fj = (u / Bk::X) % (Bk::Y + 1);
      fk = u / (Bk::X * (Bk::Y + 1));
    } else {
      const int u = w - Bk::PXF - Bk::PYF;
      pad = u >= Bk::NZF;
      t = Bk::NXF + Bk::NYF + u;
      dir = 2;
      fi = u % Bk::X;
      fj = (u / Bk::X) % Bk::Y;
      fk = u / (Bk::X * Bk::Y);
    }
    sL = sR = MIRROR;
    if (pad) {
      d0 = -1;
      return;
    }
    // right cell (the face is its lower face) and left cell
    const int ri = i0 + fi, rj = j0 + fj, rk = k0 + fk;
    const int li = ri - (dir == 0), lj = rj - (dir == 1), lk = rk - (dir == 2);
    const bool rIn = ri < g.nx && rj < g.ny && (D == 2 || rk < g.nz);
    const bool lIn = li >= 0 && lj >= 0 && lk >= 0 && li < g.nx && lj < g.ny && (D == 2 || lk < g.nz);
    // a face is needed when one of its cells is a live cell of this brick
    const bool rBrick = fi < Bk::X && fj < Bk::Y && fk < Bk::Z && rIn;
    const bool lBrick = (dir == 0 ? fi > 0 : (dir == 1 ? fj > 0 : fk > 0)) && lIn;
    const bool needed = rBrick || lBrick;
    // the side's source; a cell off the grid along dir wraps (periodic) or
    // mirrors the other side (wall)
    auto source = [&](int x, int y, int z) {
      const int n_ax = dir == 0 ? g.nx : (dir == 1 ? g.ny : g.nz);
      int pos = dir == 0 ? x : (dir == 1 ? y : z);
      const int row = row_of(x, y, z);
      if (pos < 0 || pos >= n_ax) {
        const bool low = pos < 0;
        if ((low ? g.bc[2 * dir] : g.bc[2 * dir + 1]) != 0) return MIRROR;
        pos = low ? pos + n_ax : pos - n_ax;
        if (dir == 0) x = pos;
        else if (dir == 1) y = pos;
        else z = pos;
      }
      if (row >= 0) return -(row + 2);
      return (z * g.ny + y) * g.nx + x;
    };
    if (needed) {
      sR = source(ri, rj, rk);
      sL = source(li, lj, lk);
    }
    d0 = t | (dir << 20) | (needed ? 1 << 30 : 0);
  };
  for (int w = tid; w < Bk::PF; w += BLK) describe(w, fd0[w], fdL[w], fdR[w]);
  // states of face f at point q from a side's source
  auto load_side = [&](int src, int f, int q, double *out) {
    if (src <= -2) {
      const double *r = a.ws + size_t(-src - 2) * (Shape<D, NQ>::F * Q * 5) + (f * Q + q) * 5;
#pragma unroll
      for (int v = 0; v < NV; v++) out[v] = r[v];
    } else {
      const double *p = FS + fs_base(size_t(src), Shape<D, NQ>::F * Q * NV) + size_t(f * Q + q) * NV * FSB;
#pragma unroll
      for (int v = 0; v < NV; v++) out[v] = p[size_t(v) * FSB];
    }
  };
  auto mirror_of = [&](const double *inner, unsigned m, double *out) {
#pragma unroll
    for (int v = 0; v < NV; v++) out[v] = ((m >> v) & 1u) ? -inner[v] : inner[v];
  };

#pragma unroll 1
  for (int q = 0; q < Q; q++) {
    // every face of the brick at point q, solved once
#pragma unroll 1
    for (int w = tid; w < Bk::PF; w += BLK) {
      const int d0 = fd0[w], sL = fdL[w], sR = fdR[w];
      if (d0 < 0) continue;
      const int t = d0 & 0xFFFFF, dir = (d0 >> 20) & 3;
      double Fl[NV];
#pragma unroll
      for (int v = 0; v < NV; v++) Fl[v] = 0.0;
      if (d0 >> 30) {
        double uL[NV], uR[NV];
        const int lo = 2 * dir + 1, hi = 2 * dir;  // left cell's upper face, right cell's lower face
        if (sR != MIRROR) {
          load_side(sR, hi, q, uR);
          if (sL == MIRROR) mirror_of(uR, g.negmask[2 * dir], uL);
          else load_side(sL, lo, q, uL);
        } else {
          load_side(sL, lo, q, uL);
          mirror_of(uL, g.negmask[2 * dir + 1], uR);
        }
        double sp;
        if (dir == 0) sp = riemann_points<0>(g, uL, uR, Fl);
        else if (dir == 1) sp = riemann_points<1>(g, uL, uR, Fl);
        else sp = riemann_points<2>(g, uL, uR, Fl);
        vmax = sp > vmax ? sp : vmax;
      }
#pragma unroll
      for (int v = 0; v < NV; v++) fl[v][t] = Fl[v];
    }
    __syncthreads();
    if (live) {
      const int tx = threadIdx.x, ty = threadIdx.y, tz = threadIdx.z;
      const int xW = tx + (Bk::X + 1) * (ty + Bk::Y * tz), xE = xW + 1;
      const int yS = Bk::NXF + tx + Bk::X * (ty + (Bk::Y + 1) * tz), yN = yS + Bk::X;
      const int zB = Bk::NXF + Bk::NYF + tx + Bk::X * (ty + Bk::Y * tz), zT = zB + Bk::X * Bk::Y;
      // the reference divides each term by the spacing; multiplying by its
      // reciprocal differs by rounding only and saves 12 NV divisions
      const double w = g.wt[q / NQ] * g.wt[q % NQ];
#pragma unroll
      for (int v = 0; v < NV; v++) {
        rhs[v] += w * (fl[v][xW] - fl[v][xE]) * rdx;
        rhs[v] += w * (fl[v][yS] - fl[v][yN]) * rdy;
        rhs[v] += w * (fl[v][zB] - fl[v][zT]) * rdz;
      }
    }
    __syncthreads();
  }

  const bool write = !a.sliceWrite || a.sliceWrite[slice] != 0;
  if (live) rk_epilogue<NV>(a, U, c, nc, rhs, betaDt, bhatDt, write, errLoc, posLoc);
  const int bid = b;  // slice-major: the bricks of a 2D slice are one contiguous range
  const double bmax = block_max(vmax, sh, tid);
  if (tid == 0 && bmax > 0.0) atomicMax(a.vmaxBits + slice, (unsigned long long)__double_as_longlong(bmax));
  if (a.mode == RK_FSAL) {
    const double es = block_sum(errLoc, sh, tid);
    const double pm = block_min(posLoc, sh, tid);
    if (tid == 0) {
      a.errPartial[bid] = es;
      a.posPartial[bid] = pm;
    }
  }
}

}  // namespace dev
}  // namespace kfvm
