// Path pool kernels over dense grids with the trilinear filter or 2^32 voxels and more.
#include "path_pool.hpp"

namespace crvpt {
CRVPT_INSTANTIATE_POOL(DenseAccess)
}  // namespace crvpt
