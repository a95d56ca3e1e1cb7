// Path pool kernels over NanoVDB grids below 4 GiB with axis-aligned voxels, trilinear filter.
#include "path_pool.hpp"

namespace crvpt {
CRVPT_INSTANTIATE_POOL(NanoAccessNarrow)
}  // namespace crvpt
