// GLM-MHD kernel instantiation for dimension 2, 3 Gauss points per face direction.
#include "launch_impl.hpp"

namespace kfvm {
template struct LaunchMhd<2, 3>;
}  // namespace kfvm
