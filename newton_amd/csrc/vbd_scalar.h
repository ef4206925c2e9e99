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

#ifdef __HIP__
VBD_SCALAR float exp2_hw(float x) { return __builtin_amdgcn_exp2f(x); }
VBD_SCALAR float rcp_hw(float x) { return __builtin_amdgcn_rcpf(x); }  // results below 2^-126 are 0
VBD_SCALAR float clamp_hw(float x, float lo, float hi) { return __builtin_amdgcn_fmed3f(x, lo, hi); }
#else
VBD_SCALAR float exp2_hw(float x) { return exp2f(x); }
VBD_SCALAR float rcp_hw(float x) { return 1.0f / x < FLT_MIN ? 0.0f : 1.0f / x; }
VBD_SCALAR float clamp_hw(float x, float lo, float hi) { return fminf(fmaxf(x, lo), hi); }
#endif

// 1 / (1 + exp(-z)) to about an ulp, as expf and an IEEE division give it, in 11 instructions instead of 40: exp2 of
// -z log2(e) with the product's low part put back, and the reciprocal with one Newton step.  z is held within
// [-88, 88] before the product is split, so the low part stays an ulp of it and nothing overflows; at the lower end
// the reciprocal, under 2^-126, is 0 and stays 0 through the Newton step, at the upper the sigmoid is 1.  NaN may come
// out as a number: SiLU and its derivative multiply by z.  (The result's zero selected below the range instead:
// training step of 16,384 rows 51.7 us, 50.8 us so.)
VBD_SCALAR float sigmoid_short(float z) {
    const float l2e = 1.44269502f, l2e_lo = 1.92596299e-8f, ln2 = 0.693147182f;  // log2(e) in two parts
    const float x = clamp_hw(z, -88.0f, 88.0f);
    const float p = -x * l2e;
    const float lo = __builtin_fmaf(-x, l2e, -p) - x * l2e_lo;
    const float e = exp2_hw(p);
    const float d = 1.0f + __builtin_fmaf(e * ln2, lo, e);
    const float r = rcp_hw(d);
    return __builtin_fmaf(__builtin_fmaf(-d, r, 1.0f), r, r);
}

}  // namespace vbd_scalar
