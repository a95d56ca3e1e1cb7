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

// a / c for the constant divisors c of the default sky, rc the rounded 1 / c: the same correction, for finite a. Equal to
// the division for every mantissa of a (host test).
CRVPT_SCALAR float divRounded(float a, float c, float rc) {
    const float q = a * rc;
    return fmaf(fmaf(-q, c, a), rc, q);
}

// x^2.4 = x^2 x^0.4 for x in [2^-4, 2] from x2 = x^2, y = x^0.4 to a few units of float, y4 = y^4 and r, about 1 / (5 y4):
// one Newton step of y^5 = x^2, in FP64 but for the correction. Within 0.501 units in the last place of the exact power
// (host test), against 1 for the library's power, which also takes the rounded exponent.
CRVPT_SCALAR float pow24From(double x2, double y, double y4, float r) {
    const float d = float(fma(-y4, y, x2)) * r;
    return float(x2 * (y + double(d)));
}

}  // namespace crvpt
