// Device powers and reciprocal square roots in FP64, straight-line code.
#pragma once

#include <hip/hip_runtime.h>

namespace ssu {
namespace {

// FP64 log2 of a positive finite x (subnormals too: the hardware frexp):
// x = m 2^e with m in [sqrt(1/2), sqrt(2)), log2 m = (2 / ln 2) atanh t with
// t = (m - 1) / (m + 1), |t| <= 0.1716, summed as t (1 + t^2/3 + t^4/5 + ... +
// t^24/25) (the next term is below 2e-20 of the sum): a few ulps, against the
// many branches of the general pow.
__device__ __forceinline__ double log2_pos(double x) {
    int e = __builtin_amdgcn_frexp_exp(x);
    double m = __builtin_amdgcn_frexp_mant(x);   // [0.5, 1)
    if (m < 0.70710678118654752440) { m *= 2.0; --e; }
    const double t = (m - 1.0) / (m + 1.0), t2 = t * t;
    double p = 1.0 / 25.0;
    p = fma(p, t2, 1.0 / 23.0);
    p = fma(p, t2, 1.0 / 21.0);
    p = fma(p, t2, 1.0 / 19.0);
    p = fma(p, t2, 1.0 / 17.0);
    p = fma(p, t2, 1.0 / 15.0);
    p = fma(p, t2, 1.0 / 13.0);
    p = fma(p, t2, 1.0 / 11.0);
    p = fma(p, t2, 1.0 / 9.0);
    p = fma(p, t2, 1.0 / 7.0);
    p = fma(p, t2, 1.0 / 5.0);
    p = fma(p, t2, 1.0 / 3.0);
    p = fma(p, t2, 1.0);
    return (double)e + (t * p) * 2.88539008177792681472;   // 2 / ln 2
}

// FP64 2^y for |y| < 2^31: y = k + f with k = rint(y), |f| <= 1/2, and
// 2^f = e^z, z = f ln 2, from the Taylor series to z^16/16! (|z| <= 0.347:
// the next term is below 1e-21), scaled by ldexp (which overflows and underflows as 2^y does).
__device__ __forceinline__ double exp2_finite(double y) {
    const double k = rint(y);
    const double z = (y - k) * 0.69314718055994530942;   // ln 2
    double p = 1.0 / 20922789888000.0;                    // 1/16!
    p = fma(p, z, 1.0 / 1307674368000.0);
    p = fma(p, z, 1.0 / 87178291200.0);
    p = fma(p, z, 1.0 / 6227020800.0);
    p = fma(p, z, 1.0 / 479001600.0);
    p = fma(p, z, 1.0 / 39916800.0);
    p = fma(p, z, 1.0 / 3628800.0);
    p = fma(p, z, 1.0 / 362880.0);
    p = fma(p, z, 1.0 / 40320.0);
    p = fma(p, z, 1.0 / 5040.0);
    p = fma(p, z, 1.0 / 720.0);
    p = fma(p, z, 1.0 / 120.0);
    p = fma(p, z, 1.0 / 24.0);
    p = fma(p, z, 1.0 / 6.0);
    p = fma(p, z, 0.5);
    p = fma(p, z, 1.0);
    p = fma(p, z, 1.0);
    return ldexp(p, (int)k);
}

// x^a for finite x > 0 in FP64, |a log2 x| < 2^31: 2^(a log2 x)
__device__ __forceinline__ double dpow64(double x, double a) { return exp2_finite(a * log2_pos(x)); }

// 1 / sqrt(x) for normal x > 0 in FP64: the hardware FP64 reciprocal square
// root approximation (5.2e-8 relative at most, measured over 1e-30..1e30)
// refined by STEPS Newton steps r += r (1 - x r^2) / 2, each of which squares
// the relative error (one step: 4.1e-15; two: FP64 rounding).  Straight-line
// code, no branch.
template <int STEPS> __device__ __forceinline__ double rsqrt_nr(double x) {
    double r = __builtin_amdgcn_rsq(x);
#pragma unroll
    for (int i = 0; i < STEPS; ++i) {
        const double e = fma(-x * r, r, 1.0);
        r = fma(0.5 * r, e, r);
    }
    return r;
}

}  // namespace
}  // namespace ssu
