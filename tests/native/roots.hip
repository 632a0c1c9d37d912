// roots.hip — rcp_exact, sqrt_exact and quot_exact (polyred_amd/csrc/roots.hpp)
// over every float32 mantissa on the GPU, against the correctly rounded results.
// Those come from float64: a quotient of two float32 and a root of one are
// further from every float32 rounding boundary (2^-50 relative) than float64's
// rounding moves them.
#include "roots.hpp"

#include <stdint.h>

namespace {

struct Bad {
    unsigned long long n;
    uint32_t a, x;  // one of them
};
__device__ float of(uint32_t mant, int e) { return __uint_as_float((uint32_t)(e + 127) << 23 | mant); }
__device__ void check(Bad* bad, float got, float want, float a, float x) {
    if (__float_as_uint(got) == __float_as_uint(want)) return;
    atomicAdd(&bad->n, 1ull);
    bad->a = __float_as_uint(a), bad->x = __float_as_uint(x);
}
// A thread a mantissa (2^23 threads), over the exponents [e0, e1).
__global__ void k_rcp(int e0, int e1, Bad* bad) {
    const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
    for (int e = e0; e < e1; e++) {
        const float x = of(m, e);
        check(bad, prh::rcp_exact(x), (float)(1.0 / (double)x), 1.0f, x);
        check(bad, prh::rcp_exact(-x), (float)(-1.0 / (double)x), 1.0f, -x);
    }
}
__global__ void k_sqrt(int e0, int e1, Bad* bad) {
    const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
    for (int e = e0; e < e1; e++) {
        const float x = of(m, e);
        check(bad, prh::sqrt_exact(x), (float)__builtin_sqrt((double)x), 0.0f, x);
    }
}
// A thread a divisor's mantissa, `n` numerators each: mixed from the seed, and
// those next to a multiple of the divisor's half units (the hardest quotients).
__global__ void k_quot(int n, uint32_t seed, Bad* bad) {
    const uint32_t m = blockIdx.x * blockDim.x + threadIdx.x;
    uint32_t s = m * 2654435761u ^ seed;
    for (int k = 0; k < n; k++) {
        s ^= s << 13, s ^= s >> 17, s ^= s << 5;
        const float x = of(m, (int)(s >> 25) % 81 - 40), r = prh::rcp_exact(x);
        s ^= s << 13, s ^= s >> 17, s ^= s << 5;
        const float a = of(s & 0x7fffffu, (int)(s >> 24) % 81 - 40);
        check(bad, prh::quot_exact(a, x, r), (float)((double)a / (double)x), a, x);
        check(bad, prh::quot_exact(-a, x, r), (float)(-(double)a / (double)x), -a, x);
        // a quotient's midpoint times the divisor, rounded to a numerator
        const double q = (double)of(s & 0x7fffffu, 0) * (1.0 + 0x1p-24);
        const float b = (float)(q * (double)x);
        check(bad, prh::quot_exact(b, x, r), (float)((double)b / (double)x), b, x);
    }
}

}  // namespace

// which: 0 reciprocals, 1 roots (exponents [a, b)), 2 quotients (a numerators a
// divisor, seed b).  out: the number of wrong results and one's operands.
extern "C" int roots_check(int which, int a, int b, unsigned long long* n, uint32_t* one) {
    Bad* d = nullptr;
    Bad h{};
    if (hipMalloc((void**)&d, sizeof(Bad)) != hipSuccess) return 1;
    hipError_t e = hipMemcpy(d, &h, sizeof h, hipMemcpyHostToDevice);
    const dim3 grid((1u << 23) / 256), block(256);
    if (e == hipSuccess) {
        if (which == 0) hipLaunchKernelGGL(k_rcp, grid, block, 0, nullptr, a, b, d);
        else if (which == 1) hipLaunchKernelGGL(k_sqrt, grid, block, 0, nullptr, a, b, d);
        else hipLaunchKernelGGL(k_quot, grid, block, 0, nullptr, a, (uint32_t)b, d);
        e = hipGetLastError();
    }
    if (e == hipSuccess) e = hipMemcpy(&h, d, sizeof h, hipMemcpyDeviceToHost);
    (void)hipFree(d);
    *n = h.n, one[0] = h.a, one[1] = h.x;
    return e == hipSuccess ? 0 : 2;
}
