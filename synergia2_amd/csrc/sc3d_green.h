// sc3d_green.h -- the reference's Green's functions, evaluated pointwise on
// the device (space_charge_3d_open_hockney.cc:136-348): the integrated
// (linear) Green's function of alg_g2_linear and the point-charge one of
// alg_g2_pointlike, with their origin values G000.  Shared by the spectrum
// passes (sc3d_fft.hip) and the index-decomposition patches
// (sc3d_quirk.hip), so both evaluate the same arithmetic.
#pragma once

#include "sc3d_exact.h"

namespace sc3d {

// G000 of the two functions (space_charge_3d_open_hockney.cc:165,265-270).
__device__ __forceinline__ double green_g000(int green_fn, double hx, double hy, double hz)
{
    if (green_fn == SC3D_GREEN_LINEAR) {
        double rr = hx * hx + hy * hy;
        double r1 = sqrt(hx * hx + hy * hy + hz * hz);
        return (2.0 / rr) * (hz * r1 + rr * log((hz + r1) / sqrt(rr)) - hz * hz);
    }
    return 2.8 / fmin(hx, fmin(hy, hz));
}

// log(r), r >= 1, to about 1 ulp.  Up to 1.25: with f = r - 1 (exact) and
// s = f / (2 + f), log(1 + f) = 2 atanh(s) and f - 2 s = s f, so it is
// f - s (f - 2 s^2 h(s^2)), h(w) = sum w^k / (2k + 3) as a polynomial fitted
// on s <= 1/9 (error 1.5e-18 of the logarithm).
__device__ __forceinline__ double log_above_one(double r)
{
    if (r > 1.25) return log(r);
    const double f = r - 1.0;
    const double s = f * rcp_near(2.0 + f);
    const double w = s * s;
    double h = 0.07944349896236011244;
    h = __builtin_fma(h, w, 0.09087385278226896519);
    h = __builtin_fma(h, w, 0.11111133738640772574);
    h = __builtin_fma(h, w, 0.14285714220134911617);
    h = __builtin_fma(h, w, 0.20000000000069450525);
    h = __builtin_fma(h, w, 0.33333333333333321423);
    return __builtin_fma(-s, __builtin_fma(-2.0 * w, h, f), f);
}

// The spectrum's first pass is bound by this function: 400 instructions a
// point, two logarithms, three square roots and two divisions in their general
// forms.  Beyond z = hz every argument is positive and in range, so it takes
// the short forms (the roots keep their bits, the quotients almost always; the
// logarithm is as close, and enters multiplied by about hz / r).  Measured (k_green_x, us):
// 128x128x256 FP32 64.6 -> 45.3, 64x64x128 FP64 15.9 -> 13.1, 32x32x64 FP64
// 9.2 -> 7.6.
__device__ __forceinline__ double green_linear(double x, double y, double z, double hx, double hy,
                                               double hz)
{
    const double rr = x * x + y * y;
    const double epsz = 1e-12 * hz;
    // z >= 0 here, so of the reference's branches (:294-326) only these three
    // are reachable; the z < -hz and |z + hz| < epsz ones never are.
    const bool near = fabs(z) < epsz || fabs(z - hz) < epsz || !(z > hz);
    if (!near && hz > 1.0e-100 && rr < 1.0e200 && z < 1.0e100) {
        const double s_rr_0 = sqrt_normal(rr + z * z);
        const double s_rr_n = sqrt_normal(rr + (z - hz) * (z - hz));
        const double s_rr_p = sqrt_normal(rr + (z + hz) * (z + hz));
        const double G = 2.0 * s_rr_0 - s_rr_n - s_rr_p;
        const double r1 = div_normal(s_rr_0 + z, s_rr_n + z - hz);
        const double r2 = div_normal(s_rr_p + z + hz, s_rr_0 + z);
        const double T1 = (hz - z) * log_above_one(r1);
        const double T2 = (hz + z) * log_above_one(r2);
        return G + (T1 + T2);
    }
    double s_rr_0 = sqrt(rr + z * z);
    double s_rr_n = sqrt(rr + (z - hz) * (z - hz));
    double s_rr_p = sqrt(rr + (z + hz) * (z + hz));
    double G = 2.0 * s_rr_0 - s_rr_n - s_rr_p;
    double T1, T2, r1, r2;
    if (fabs(z) < epsz) {
        if (fabs(x) + fabs(y) < 2. * epsz) {
            G += hz * green_g000(SC3D_GREEN_LINEAR, hx, hy, hz);
        } else {
            r1 = (sqrt(hz * hz + rr) + hz) / sqrt(rr);
            G += 2.0 * hz * log(r1);
        }
    } else if (fabs(z - hz) < epsz) {
        r1 = (s_rr_p + z + hz) / (s_rr_0 + z);
        T1 = (hz + z) * log(r1);
        G += T1;
    } else if (z > hz) {
        r1 = (s_rr_0 + z) / (s_rr_n + z - hz);
        T1 = (hz - z) * log(r1);
        r2 = (s_rr_p + z + hz) / (s_rr_0 + z);
        T2 = (hz + z) * log(r2);
        G += T1 + T2;
    }
    return G;
}

// The value the reference writes for the point with coordinates (x, y, z)
// >= 0 (z already folded: (Dz - iz) * hz above the middle plane for the
// linear function); pointlike: G000 at the origin, 1/r elsewhere.
__device__ __forceinline__ double green_value(int green_fn, double x, double y, double z,
                                              double hx, double hy, double hz)
{
    if (green_fn == SC3D_GREEN_LINEAR) return green_linear(x, y, z, hx, hy, hz);
    return (x == 0.0 && y == 0.0 && z == 0.0) ? green_g000(green_fn, hx, hy, hz)
                                              : 1.0 / sqrt(x * x + y * y + z * z);
}

}  // namespace sc3d
