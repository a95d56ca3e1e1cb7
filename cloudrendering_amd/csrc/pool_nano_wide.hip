// Path pool kernels over any NanoVDB grid (64-bit offsets, full index map).
#include "path_pool.hpp"

namespace crvpt {
CRVPT_INSTANTIATE_POOL(NanoAccess)
}  // namespace crvpt
