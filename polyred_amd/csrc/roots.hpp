// roots.hpp — reciprocals, quotients and roots without the compiler's scaling
// and special cases, for operands in a range in which no step over- or
// underflows; the callers take the plain ones outside.  Each is the correctly
// rounded result, as the plain one: the reciprocal and the root by the
// hardware's estimate (1 ulp) and one residual step (Markstein 1990), the
// quotient by a residual step from the correctly rounded reciprocal.  That the
// step is exact is a property of this hardware's estimates (with the other
// faithful estimate of some mantissas it would not be):
// tests/test_gpu_roots.py runs all of them through it.
#pragma once

#include <hip/hip_runtime.h>

namespace prh {

__device__ __forceinline__ float rcp_exact(float x) {  // 1 / x, 2^-100 <= |x| < 2^100
    const float y = __builtin_amdgcn_rcpf(x);
    return __builtin_fmaf(__builtin_fmaf(-x, y, 1.0f), y, y);
}
// a / x with r = rcp_exact(x); a and a / x from 2^-100 to 2^100, or 0
__device__ __forceinline__ float quot_exact(float a, float x, float r) {
    const float q = a * r;
    return __builtin_fmaf(__builtin_fmaf(-x, q, a), r, q);
}
__device__ __forceinline__ float sqrt_exact(float d) {  // sqrt(d), 2^-64 <= d < 2^64
    const float r = __builtin_amdgcn_rsqf(d), g = d * r;
    return __builtin_fmaf(__builtin_fmaf(-g, g, d), 0.5f * r, g);
}

}  // namespace prh
