// Quotients by a value that many share.  Comes after the HIP runtime's header, or
// in a host program with __device__ and __forceinline__ defined away.
#pragma once
#include <cmath>

namespace sg {

// a / d, correctly rounded, for a d that many a share: r = 1 / d.  The product
// a r is within two units in the last place, one correction makes it faithful
// and the second, whose remainder is exact, rounds as the division does
// (Markstein's theorem) while nothing leaves the normal range (a of -0 gives +0).
struct Divisor {
    double d, r;
    __device__ explicit Divisor(double v) : d(v), r(1.0 / v) {}
    __device__ static bool safe(double v) { return fabs(v) > 0x1p-60 && fabs(v) < 0x1p60; }
    __device__ __forceinline__ double operator()(double a) const {
        const double q = a * r, p = __builtin_fma(__builtin_fma(-d, q, a), r, q);
        return __builtin_fma(__builtin_fma(-d, p, a), r, p);
    }
};

}  // namespace sg
