// Definition of the dense GLM-MHD linear launcher (launch_decl.hpp), included by
// its instantiation units inst_mhd_dense_*.hip only: the unrolled products of
// nine variables take minutes to compile.
#pragma once

#include "launch_decl.hpp"

#include "stage_kernels.hpp"

namespace kfvm {

template <int D, int NQ>
hipError_t LaunchMhdDense<D, NQ>::linear(const double *U, double *FS, double *SRC, double *WI, double *thetaNew,
                                     double *spd, const double *props, const Grid &g, const double *WT,
                                     int *ppList, int *ppCount, hipStream_t s) {
  hipLaunchKernelGGL((dev::k_mhd_linear<D, NQ>), dim3(LaunchMhd<D, NQ>::bricks(g)), dim3(dev::MBox<D>::NT), 0, s, U, FS, SRC,
                     WI, thetaNew, spd, props, g, WT, ppList, ppCount);
  return hipGetLastError();
}

}  // namespace kfvm
