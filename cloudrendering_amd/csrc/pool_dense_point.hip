// Path pool kernels over dense grids below 2^32 voxels with a point filter.
#include "path_pool.hpp"

namespace crvpt {
CRVPT_INSTANTIATE_POOL(DenseAccessPoint)
}  // namespace crvpt
