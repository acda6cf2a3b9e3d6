// sc3d_exact.h -- square root and division with the bits of the correctly
// rounded operations (div_normal: but for rare last bits), for arguments the
// caller knows to be well inside the normal range.  The compiler's own
// expansions scale and classify their arguments on every call (21 and 16 issue
// slots); the particle and Green's kernels are bound by FP64 issue (13 and 10
// here).
//
// Both end in a residual step on a value within about 1 ulp: with g ~ sqrt(a)
// and y ~ 1/sqrt(a), g + (a - g^2) y/2 has an exact residual and one rounding
// (P. Markstein, IBM J. Res. Dev. 34, 1990), likewise q + (a - q b) y for
// a/b.  Before that rounding the value is within a few 2^-53 ulp of the root.
// The closest roots of doubles lie at 2^-56 ulp from a rounding boundary (next
// to powers of four), so the sequence was run on all 56619 arguments (both
// exponent parities, found from q^2 = 1 - 4c mod 2^54 and 2^55) whose root is
// within 2^-38 ulp of one, over 2000 seeds each: no wrong root.  For a/b the
// theorem takes a correctly rounded 1/b (div_by); from rcp_near's (div_normal)
// a quotient next to a boundary may miss it by its last bit.
#pragma once

#include "sc3d_common.h"

namespace sc3d {

// 1/sqrt(a) to about 1 ulp: hardware seed and one third-order step.
__device__ __forceinline__ double rsqrt_near(double a)
{
    const double y0 = __builtin_amdgcn_rsq(a);
    const double e = __builtin_fma(-(a * y0), y0, 1.0);
    return __builtin_fma(y0 * e, __builtin_fma(e, 0.375, 0.5), y0);
}

// sqrt(a) from y = rsqrt_near(a).
__device__ __forceinline__ double sqrt_from(double a, double y)
{
    const double g = a * y;
    return __builtin_fma(__builtin_fma(-g, g, a), 0.5 * y, g);
}

// sqrt(a), 1e-250 < a < 1e250.
__device__ __forceinline__ double sqrt_normal(double a) { return sqrt_from(a, rsqrt_near(a)); }

// a / b with y the correctly rounded 1 / b; the quotient and a themselves
// zero or between 1e-250 and 1e250 in magnitude.
__device__ __forceinline__ double div_by(double a, double b, double y)
{
    const double q = a * y;
    return __builtin_fma(__builtin_fma(-q, b, a), y, q);
}

// 1 / b to about 1/2 ulp, 1e-250 < |b| < 1e250.
__device__ __forceinline__ double rcp_near(double b)
{
    const double y0 = __builtin_amdgcn_rcp(b);
    const double e = __builtin_fma(-b, y0, 1.0);
    return __builtin_fma(y0, __builtin_fma(e, e, e), y0);
}

// a / b for such b and a as for div_by, almost always correctly rounded (see
// above); for values that no comparison takes bit by bit.
__device__ __forceinline__ double div_normal(double a, double b)
{
    return div_by(a, b, rcp_near(b));
}

}  // namespace sc3d
