// Scalar formulas of the kernels that the CPU tests check over their whole range (tests/scalar_check.cpp).
#pragma once

#include <cfloat>
#include <cmath>

#ifdef __HIP__
#define VBD_SCALAR __device__ __forceinline__
#else
#define VBD_SCALAR static inline
#endif

namespace vbd_scalar {

// True when the Frobenius condition number of a 3x3 block H is certainly far below 1e6, from single precision alone:
// ||adj H||_F <= ||H||_F^2 / sqrt(3), so cond <= ||H||_F^3 / (sqrt(3) |det H|); the computed determinant is
// within 5 roundings of perm|H| <= ||H||_F^3 (3e-7 of it), so |det| >= 4e-6 ||H||_F^3 bounds the condition by
// 1.6e5.  det is the computed determinant, inv_norm = 1 / ||H||_F.  A determinant that overflowed or is NaN proves
// nothing; a norm whose square overflowed gives inv_norm = 0.  An underflow of a square cannot matter to callers with
// |det| > 1e-8, which keeps ||H||_F above 2e-3.
VBD_SCALAR bool certainly_well_conditioned(float det, float inv_norm) {
    const float d = fabsf(det);
    return d <= FLT_MAX && d * inv_norm * inv_norm * inv_norm >= 4.0e-6f;
}

}  // namespace vbd_scalar
