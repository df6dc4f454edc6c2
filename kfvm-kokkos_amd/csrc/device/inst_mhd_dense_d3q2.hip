// Dense GLM-MHD linear pass for dimension 3, 2 Gauss points per face direction.
#include "launch_mhd_dense.hpp"

namespace kfvm {
template struct LaunchMhdDense<3, 2>;
}  // namespace kfvm
