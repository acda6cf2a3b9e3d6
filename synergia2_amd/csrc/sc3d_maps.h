// sc3d_maps.h -- single-particle maps of the FODO channel (drift and
// quadrupole), host+device so the design reference particle's cdt is
// computed with the identical arithmetic.
//
//   drift_unit          <- FF_algorithm::drift_unit, libFF/ff_algorithm.h:45-79
//   thin_quadrupole_unit<- libFF/ff_algorithm.h:928-936
//   yoshida6            <- libFF/ff_algorithm.h:1835-2008 (10 drifts and 9
//                          thin kicks per step; default 4 steps per slice,
//                          ff_quadrupole.h:438-441)
//   reference cdt       <- drift_impl::get_reference_cdt (ff_drift.h:68-87),
//                          quad_impl::get_reference_cdt (ff_quadrupole.h:262-300)
#pragma once

#include <hip/hip_runtime.h>

#include "../../include/sc3d_capi.h"
#include "sc3d_exact.h"

namespace sc3d {

__host__ __device__ inline void drift_unit(double& x, double xp, double& y, double yp,
                                           double& cdt, double dpop, double length,
                                           double reference_momentum, double m,
                                           double reference_cdt)
{
    const double uni = 1.0;
    const double sig = double((0.0 < length) - (length < 0.0));
    const double vl = length, vm = m, vrm = reference_momentum, vrc = reference_cdt;
    double dp = dpop + uni;
    double inv_npz = uni / sqrt(dp * dp - xp * xp - yp * yp);
    double lxpr = xp * vl * inv_npz;
    double lypr = yp * vl * inv_npz;
    double D2 = lxpr * lxpr + vl * vl + lypr * lypr;
    double p = dp * vrm;
    double E2 = p * p + vm * vm;
    double ibeta2 = E2 / (p * p);
    x = x + lxpr;
    y = y + lypr;
    cdt = cdt + sig * sqrt(D2 * ibeta2) - vrc;
}

__host__ __device__ inline void thin_quadrupole_unit(double x, double& xp, double y, double& yp,
                                                     const double* kL)
{
    const double vk0 = kL[0], vk1 = kL[1];
    xp = xp - vk0 * x + vk1 * y;
    yp = yp + vk0 * y + vk1 * x;
}

// Sixth-order composition: drifts of c[0..3], thin kicks of d[0..3] per step.
constexpr double kYoshidaDrift[4] = {0.79361246386112147294625603763,
                                     -0.206276584816439780698721319354,
                                     -0.118008867881292655922412133144,
                                     0.236949573653050744373598734219};
constexpr double kYoshidaKick[4] = {1.58722492772224294589251207526,
                                    -1.99977809735512250728995471397,
                                    -1.82324266348482825773733634154,
                                    2.29714181079092974648453380998};
constexpr int kYoshidaDrifts = 10;
constexpr int kYoshidaDriftOrder[kYoshidaDrifts] = {0, 1, 1, 2, 3, 3, 2, 1, 1, 0};
constexpr int kYoshidaKickOrder[kYoshidaDrifts] = {0, 1, 0, 2, 3, 2, 0, 1, 0, 0};  // 9 used

// The stages one after the other, for the rolled loops.
struct YoshidaStage {
    double drift, kick;
};
constexpr YoshidaStage yoshida_stage(int q)
{
    return {kYoshidaDrift[kYoshidaDriftOrder[q]], kYoshidaKick[kYoshidaKickOrder[q]]};
}
constexpr YoshidaStage kYoshidaStages[kYoshidaDrifts] = {
    yoshida_stage(0), yoshida_stage(1), yoshida_stage(2), yoshida_stage(3), yoshida_stage(4),
    yoshida_stage(5), yoshida_stage(6), yoshida_stage(7), yoshida_stage(8), yoshida_stage(9)};

// General form; rolled, so that on the device it stays out of the way of the
// fast form's registers (unrolled it set the maps kernels' count: 147 VGPRs).
__host__ __device__ inline void yoshida6_quad(double& x, double& xp, double& y, double& yp,
                                              double& cdt, double dpop, double reference_momentum,
                                              double m, double step_reference_cdt,
                                              double step_length, const double* step_strength,
                                              int steps)
{
    const double sub = step_reference_cdt * 0.1;
    for (int i = 0; i < steps; ++i) {
#pragma nounroll
        for (int q = 0; q < kYoshidaDrifts; ++q) {
            const YoshidaStage g = kYoshidaStages[q];
            drift_unit(x, xp, y, yp, cdt, dpop, g.drift * step_length, reference_momentum, m, sub);
            if (q == kYoshidaDrifts - 1) break;
            const double kL[2] = {g.kick * step_strength[0], g.kick * step_strength[1]};
            thin_quadrupole_unit(x, xp, y, yp, kL);
        }
    }
}

// A slice as the kernels take it: a quadrupole's per-step strength
// k*(length/steps) (ff_quadrupole.h:446), step length length/steps and step
// reference cdt ref_cdt/steps (ff_quadrupole.h:466-468) are formed once on the
// host (the same IEEE operations); a drift is one step.
struct PreparedSlice {
    int32_t kind;   // SC3D_MAP_*
    int32_t steps;
    double length;  // of one step
    double k[2];    // normal and skew thin-kick strength of one step
    double ref_cdt; // of one step
};
static_assert(sizeof(PreparedSlice) == sizeof(sc3d_map_slice), "layout");

inline PreparedSlice prepare_slice(const sc3d_map_slice& s)
{
    PreparedSlice q{};
    q.kind = s.kind;
    q.steps = s.kind == SC3D_MAP_DRIFT ? 1 : s.yoshida_steps;
    if (s.kind == SC3D_MAP_DRIFT) {
        q.length = s.length;
        q.ref_cdt = s.ref_cdt;
    } else {
        q.length = s.length / q.steps;
        q.k[0] = s.k1 * (s.length / q.steps);
        q.k[1] = s.k1s * (s.length / q.steps);
        q.ref_cdt = s.ref_cdt / q.steps;
    }
    return q;
}

// One slice applied to one particle.
__host__ __device__ inline void apply_slice(const PreparedSlice& s, double& x, double& xp,
                                            double& y, double& yp, double& cdt, double dpop,
                                            double ref_p, double m)
{
    if (s.kind == SC3D_MAP_DRIFT)
        drift_unit(x, xp, y, yp, cdt, dpop, s.length, ref_p, m, s.ref_cdt);
    else
        yoshida6_quad(x, xp, y, yp, cdt, dpop, ref_p, m, s.ref_cdt, s.length, s.k, s.steps);
}

// Map program passed by value to kernels (no device allocation).
struct MapProgram {
    PreparedSlice s[SC3D_MAX_SLICES];
    int32_t n;
    double ref_p, mass;
};

// ---------------------------------------------------------------------------
// The same drifts with fewer instructions.  The maps are bound by FP64 issue:
// drift_unit's two correctly rounded square roots and its division cost about
// 78 VALU instructions per drift and thin kick, most of them scaling and
// special-case handling.  Here one reciprocal-square-root seed serves all
// three (38 instructions), and the results are the same bits:
//   y  ~ 1/sqrt(a), a = dp^2 - x'^2 - y'^2: hardware seed, one third-order
//      step, about 1 ulp;
//   s  = sqrt(a) from y (sc3d_exact.h);
//   1/s = y + y (1 - s y), exact residual, the same reference; it can miss
//      when s has an all-ones significand, which `ones` records;
//   the path length sqrt(D2/beta^2) equals |l| C / s, C = dp/beta, up to a few
//      ulp: that is its seed, and s/(2 |l| C) the slope, for one residual step.
//      Signed by l, so no separate sign multiplication.
// The last step needs |l| C / s accurate to a few ulp, so a in [1/2, 2] (no
// cancellation) and 1/beta^2 away from 1 (at 1 and |l| near a power of two
// D2/beta^2 comes next to a power of four, where one residual step cannot
// decide the rounding).  A wavefront with a particle outside takes the rolled
// form for all its particles, whose path length has a square root of its own
// (any a >= 2^-100); what that form cannot hold either (a <= 0, NaN, `ones`)
// takes drift_unit.
// Measured (4e6 particles, mean over the 10 steps of an O-F-O-D cell, 6
// quadrupole slices among them): maps pass 266 -> 172 us, kick with maps fused
// (whole step) 449 -> 364 us; a step of drifts alone stays at 54 us, its
// 89 bytes per particle at 6.6 TB/s.  Four wavefronts per SIMD (<= 128 VGPRs,
// no spills) need one particle per thread: the grid-stride loop's pointers
// took the kernel to 156 VGPRs.
// ---------------------------------------------------------------------------
constexpr int32_t kHighOfHalf = 0x3fe00000;  // high word of 0.5
constexpr int32_t kHighOfTiny = 0x39b00000;  // ... of 2^-100
constexpr double kNearLight = 1.0 + 1.0e-6;  // 1/beta^2, see above

struct FastDrift {
    double dp2, ibeta2, c, half_rc;  // (1+dp/p)^2, 1/beta^2, C, 0.5 / C
    int32_t a_low;                   // smallest high word of a
    uint32_t ones;                   // largest low word of sqrt(a)
};

// Whether the slices of a program may take the fast form (the range keeps
// every residual of the path length normal).
__device__ __forceinline__ bool fast_slice(const PreparedSlice& s)
{
    const double l = fabs(s.length);
    return (l > 1.0e-60 && l < 1.0e60) || (s.kind == SC3D_MAP_DRIFT && l == 0.0);
}

__device__ __forceinline__ bool fast_begin(FastDrift& f, double dpop, double ref_p, double m)
{
    const double dp = dpop + 1.0;
    const double p = dp * ref_p;
    const double E2 = p * p + m * m;
    f.ibeta2 = E2 / (p * p);
    f.dp2 = dp * dp;
    f.c = dp * sqrt(f.ibeta2);
    f.half_rc = 0.5 / f.c;
    f.a_low = INT32_MAX;
    f.ones = 0u;
    return dp > 0.0 && f.dp2 <= 1.0e60 && f.ibeta2 >= 1.0 && f.ibeta2 < 1.0e12;
}

__device__ __forceinline__ double fast_a(FastDrift& f, double xp, double yp)
{
    const double a = f.dp2 - xp * xp - yp * yp;
    f.a_low = min(f.a_low, int32_t(__double_as_longlong(a) >> 32));
    return a;
}

// drift_unit over length l (l2 = l*l); kl ~ l C, hl ~ 1 / (2 l C).  OWN_ROOT:
// the path length by a square root of its own (kl, hl unused).
template <bool OWN_ROOT>
__device__ __forceinline__ void fast_drift(FastDrift& f, double& x, double xp, double& y,
                                           double yp, double& cdt, double l, double l2, double kl,
                                           double hl, double ref_cdt)
{
    const double a = fast_a(f, xp, yp);
    const double yr = rsqrt_near(a);
    const double s = sqrt_from(a, yr);
    f.ones = max(f.ones, uint32_t(__double_as_longlong(s)));
    const double inv_npz = __builtin_fma(yr, __builtin_fma(-s, yr, 1.0), yr);
    const double lxpr = xp * l * inv_npz;
    const double lypr = yp * l * inv_npz;
    const double D2 = lxpr * lxpr + l2 + lypr * lypr;
    const double A = D2 * f.ibeta2;
    double path;
    if (OWN_ROOT) {
        path = __builtin_copysign(sqrt_normal(A), l);
    } else {
        const double t = kl * inv_npz;
        path = __builtin_fma(__builtin_fma(-t, t, A), s * hl, t);
    }
    x = x + lxpr;
    y = y + lypr;
    cdt = cdt + path - ref_cdt;
}

// A wavefront-uniform value in scalar registers.
__device__ __forceinline__ double uniform_f64(double v)
{
    const long long b = __double_as_longlong(v);
    const unsigned lo = unsigned(__builtin_amdgcn_readfirstlane(int(b)));
    const unsigned hi = unsigned(__builtin_amdgcn_readfirstlane(int(b >> 32)));
    return __longlong_as_double((long long)((uint64_t(hi) << 32) | lo));
}

// yoshida6_quad by fast drifts.  With no skew strength its products are +-0,
// which a finite sum does not feel, and a coordinate that is not finite makes a
// so as well (the general form).
__device__ __forceinline__ void fast_quad(FastDrift& f, const PreparedSlice& s, double& x,
                                          double& xp, double& y, double& yp, double& cdt)
{
    const double r = f.half_rc / s.length, kc = f.c * s.length;
    const double sub = uniform_f64(s.ref_cdt * 0.1);
    double l[4], l2[4], kl[4], hl[4], k[4];
#pragma unroll
    for (int j = 0; j < 4; ++j) {
        l[j] = uniform_f64(kYoshidaDrift[j] * s.length);
        l2[j] = uniform_f64(l[j] * l[j]);
        kl[j] = kYoshidaDrift[j] * kc;
        hl[j] = (1.0 / kYoshidaDrift[j]) * r;
        k[j] = uniform_f64(kYoshidaKick[j] * s.k[0]);
    }
    for (int i = 0; i < s.steps; ++i) {
#pragma unroll
        for (int q = 0; q < kYoshidaDrifts; ++q) {
            const int j = kYoshidaDriftOrder[q], n = kYoshidaKickOrder[q];
            fast_drift<false>(f, x, xp, y, yp, cdt, l[j], l2[j], kl[j], hl[j], sub);
            if (q < kYoshidaDrifts - 1) {
                xp = xp - k[n] * x;
                yp = yp + k[n] * y;
            }
        }
    }
}

// The same with a skew strength, next to the speed of light and for wide
// bunches; rolled: a second unrolled form does not fit the 128 registers (740 us
// where the unrolled one takes 505 and the general one 1000; 4e6 particles,
// O-F-O-D).
__device__ __forceinline__ void fast_quad_rolled(FastDrift& f, const PreparedSlice& s, double& x,
                                                 double& xp, double& y, double& yp, double& cdt)
{
    const double sub = s.ref_cdt * 0.1;
    for (int i = 0; i < s.steps; ++i) {
#pragma nounroll
        for (int q = 0; q < kYoshidaDrifts; ++q) {
            const YoshidaStage g = kYoshidaStages[q];
            const double l = uniform_f64(g.drift * s.length);
            fast_drift<true>(f, x, xp, y, yp, cdt, l, l * l, 0.0, 0.0, sub);
            if (q == kYoshidaDrifts - 1) break;
            const double kL[2] = {g.kick * s.k[0], g.kick * s.k[1]};
            thin_quadrupole_unit(x, xp, y, yp, kL);
        }
    }
}

__device__ __forceinline__ void fast_slice_apply(FastDrift& f, const PreparedSlice& s,
                                                 bool rolled, double& x, double& xp, double& y,
                                                 double& yp, double& cdt)
{
    const double l = s.length;
    if (s.kind == SC3D_MAP_DRIFT) {
        if (l == 0.0) {
            fast_a(f, xp, yp);
            x = x + xp * l;
            y = y + yp * l;
            cdt = cdt + 0.0 - s.ref_cdt;
        } else if (rolled)
            fast_drift<true>(f, x, xp, y, yp, cdt, l, l * l, 0.0, 0.0, s.ref_cdt);
        else
            fast_drift<false>(f, x, xp, y, yp, cdt, l, l * l, l * f.c, f.half_rc / l, s.ref_cdt);
    } else if (rolled || s.k[1] != 0.0) {
        fast_quad_rolled(f, s, x, xp, y, yp, cdt);
    } else {
        fast_quad(f, s, x, xp, y, yp, cdt);
    }
}

// The whole program on one particle: the fast form; in a wavefront with a
// particle out of its range (tested after every slice) the rolled form from the
// start state, which `again` brings back (re-read rather than held: 10
// registers over the fast loop); the general form for what is left.  4e6
// particles, O-F-O-D, one at |x'| = 0.8 per wavefront: 742 us (515 without; the
// whole fast program and then the general one 1063).
template <typename Again>
__device__ __forceinline__ void apply_program(const MapProgram& prog, double& x, double& xp,
                                              double& y, double& yp, double& cdt, double dpop,
                                              Again&& again)
{
    bool fast = true;  // uniform
    for (int k = 0; k < prog.n; ++k) fast = fast && fast_slice(prog.s[k]);
    if (fast) {
        FastDrift f;
        if (fast_begin(f, dpop, prog.ref_p, prog.mass)) {
            // uniform over the lanes in here
            bool rolled = __any(f.ibeta2 <= kNearLight || f.dp2 > 2.0);
            int k;
            for (;;) {
                for (k = 0; k < prog.n; ++k) {
                    fast_slice_apply(f, prog.s[k], rolled, x, xp, y, yp, cdt);
                    if (!rolled && __any(f.a_low < kHighOfHalf)) break;
                }
                if (k == prog.n || __any(f.a_low < kHighOfTiny)) break;
                again();
                f.a_low = INT32_MAX;
                f.ones = 0u;
                rolled = true;
            }
            const bool held = k == prog.n && f.a_low >= kHighOfTiny && f.ones != 0xffffffffu;
            if (held) return;
            again();
        }
    }
    for (int k = 0; k < prog.n; ++k)
        apply_slice(prog.s[k], x, xp, y, yp, cdt, dpop, prog.ref_p, prog.mass);
}

// i, opaque to the compiler: a load at it is not merged with an earlier one.
__device__ __forceinline__ int64_t reread_index(int64_t i)
{
    asm volatile("" : "+v"(i));
    return i;
}

}  // namespace sc3d
