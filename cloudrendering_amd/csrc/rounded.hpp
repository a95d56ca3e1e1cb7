// Scalar formulas whose rounding is relied on, in plain C++ so that the host tests compile the same lines as the
// kernels.
#pragma once

#include <cmath>

#ifdef __HIP__
#define CRVPT_SCALAR __host__ __device__ __forceinline__
#else
#define CRVPT_SCALAR inline
#endif

namespace crvpt {

// a / c for a >= 0 from rc, the rounded 1 / c, with one correction of the product: the rounded quotient (equal to the
// division's in all 2^27 random pairs tried), three operations where c serves many a, and a test that keeps an infinite
// product, which the correction would turn into NaN.
CRVPT_SCALAR float quotient(float a, float c, float rc) {
    const float q = a * rc;
    const float r = fmaf(fmaf(-q, c, a), rc, q);
    return q > 3.402823466e38f ? q : r;
}

}  // namespace crvpt
