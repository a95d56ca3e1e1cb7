// Path pool kernels over NanoVDB grids below 4 GiB with axis-aligned voxels and a point filter.
#include "path_pool.hpp"

namespace crvpt {
CRVPT_INSTANTIATE_POOL(NanoAccessNarrowPoint)
}  // namespace crvpt
