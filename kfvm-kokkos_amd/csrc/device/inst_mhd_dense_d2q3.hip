// Dense GLM-MHD linear pass for dimension 2, 3 Gauss points per face direction.
#include "launch_mhd_dense.hpp"

namespace kfvm {
template struct LaunchMhdDense<2, 3>;
}  // namespace kfvm
