// sc3d_dft.h -- short DFTs in registers (forward sign -1, INV: +1, both
// unnormalised) and twiddle products, shared by the power-of-two passes
// (sc3d_fft.hip) and the passes of other lengths (sc3d_fft_any.hip).
#pragma once

#include "sc3d_common.h"

namespace sc3d {

// a * w, w = e^(-i t) (inverse: e^(+i t)), from c = cos t and s = sin t
// (fused multiply-adds: the build contracts nothing by itself)
template <bool INV, typename T2, typename F>
__device__ __forceinline__ T2 rotate(T2 a, F c, F s)
{
    T2 o;
    if (!INV) { o.x = fma(a.x, c, a.y * s); o.y = fma(a.y, c, -(a.x * s)); }
    else      { o.x = fma(a.x, c, -(a.y * s)); o.y = fma(a.y, c, a.x * s); }
    return o;
}

// a * w for a twiddle w (INV: a * conj(w)), fused multiply-adds
template <bool INV, typename T2>
__device__ __forceinline__ T2 twmul(T2 a, T2 w)
{
    T2 o;
    if (!INV) { o.x = fma(a.x, w.x, -(a.y * w.y)); o.y = fma(a.x, w.y, a.y * w.x); }
    else      { o.x = fma(a.x, w.x, a.y * w.y);    o.y = fma(a.y, w.x, -(a.x * w.y)); }
    return o;
}

// Prime lengths: cos and sin of 2 pi k / R, k = 1..(R-1)/2.
template <int R> struct PrimeRoots;
template <> struct PrimeRoots<3> {
    static constexpr double c[1] = {-0.5};
    static constexpr double s[1] = {0.86602540378443864676};
};
template <> struct PrimeRoots<5> {
    static constexpr double c[2] = {0.3090169943749474241, -0.8090169943749474241};
    static constexpr double s[2] = {0.95105651629515357212, 0.58778525229247312917};
};
template <> struct PrimeRoots<7> {
    static constexpr double c[3] = {0.62348980185873353053, -0.22252093395631440429,
        -0.90096886790241912624};
    static constexpr double s[3] = {0.78183148246802980871, 0.97492791218182360702,
        0.43388373911755812048};
};
template <> struct PrimeRoots<11> {
    static constexpr double c[5] = {0.84125353283118116886, 0.41541501300188642553,
        -0.14231483827328514044, -0.65486073394528506406, -0.95949297361449738989};
    static constexpr double s[5] = {0.54064081745559758211, 0.90963199535451837141,
        0.98982144188093273238, 0.75574957435425828377, 0.28173255684142969771};
};
template <> struct PrimeRoots<13> {
    static constexpr double c[6] = {0.8854560256532098959, 0.56806474673115580251,
        0.12053668025532305335, -0.35460488704253562597, -0.74851074817110109863,
        -0.97094181742605202716};
    static constexpr double s[6] = {0.46472317204376854566, 0.82298386589365639458,
        0.9927088740980539928, 0.93501624268541482344, 0.66312265824079520238,
        0.23931566428755776715};
};
// Length-R DFT, R odd prime: with a_j = v_j + v_{R-j} and b_j = v_j - v_{R-j},
// X_k = v_0 + sum_j a_j cos(2 pi jk/R) -+ i sum_j b_j sin(2 pi jk/R) and X_{R-k}
// with the other sign.
template <int R, bool INV, typename T2>
__device__ __forceinline__ void dft_prime(T2* v)
{
    using F = decltype(v[0].x);
    constexpr int H = (R - 1) / 2;
    T2 a[H], b[H];
    T2 sum = v[0];
#pragma unroll
    for (int j = 1; j <= H; ++j) {
        a[j - 1].x = v[j].x + v[R - j].x;
        a[j - 1].y = v[j].y + v[R - j].y;
        b[j - 1].x = v[j].x - v[R - j].x;
        b[j - 1].y = v[j].y - v[R - j].y;
        sum.x += a[j - 1].x;
        sum.y += a[j - 1].y;
    }
#pragma unroll
    for (int k = 1; k <= H; ++k) {
        T2 e = v[0], o;
        o.x = F(0);
        o.y = F(0);
#pragma unroll
        for (int j = 1; j <= H; ++j) {
            const int m = (j * k) % R, n = m <= H ? m : R - m;
            const F c = F(PrimeRoots<R>::c[n - 1]);
            const F s = m <= H ? F(PrimeRoots<R>::s[n - 1]) : -F(PrimeRoots<R>::s[n - 1]);
            e.x = fma(a[j - 1].x, c, e.x);
            e.y = fma(a[j - 1].y, c, e.y);
            o.x = fma(b[j - 1].x, s, o.x);
            o.y = fma(b[j - 1].y, s, o.y);
        }
        T2 p, q;  // e - i o, e + i o
        p.x = e.x + o.y; p.y = e.y - o.x;
        q.x = e.x - o.y; q.y = e.y + o.x;
        v[k] = INV ? q : p;
        v[R - k] = INV ? p : q;
    }
    v[0] = sum;
}

// Inverse of a modulo b (coprime, small).
constexpr int mod_inverse(int a, int b)
{
    for (int x = 1; x < b; ++x)
        if (a * x % b == 1) return x;
    return 1;
}

template <int R, bool INV, typename T2> __device__ __forceinline__ void dft_small(T2* v);

// Length A*B, A and B coprime, without twiddles (Good 1958, Thomas 1963):
// inputs n = (B n1 + A n2) mod R, outputs k with k = k1 mod A, k = k2 mod B.
template <int A, int B, bool INV, typename T2>
__device__ __forceinline__ void dft_coprime(T2* v)
{
    constexpr int R = A * B;
    T2 t[A][B];
#pragma unroll
    for (int n2 = 0; n2 < B; ++n2) {
        T2 u[A];
#pragma unroll
        for (int n1 = 0; n1 < A; ++n1) u[n1] = v[(B * n1 + A * n2) % R];
        dft_small<A, INV>(u);
#pragma unroll
        for (int k1 = 0; k1 < A; ++k1) t[k1][n2] = u[k1];
    }
#pragma unroll
    for (int k1 = 0; k1 < A; ++k1) {
        dft_small<B, INV>(t[k1]);
#pragma unroll
        for (int k2 = 0; k2 < B; ++k2)
            v[(k1 * B * mod_inverse(B, A) + k2 * A * mod_inverse(A, B)) % R] = t[k1][k2];
    }
}

template <int R, bool INV, typename T2>
__device__ __forceinline__ void dft_small(T2* v)
{
    if constexpr (R == 3 || R == 5 || R == 7 || R == 11 || R == 13) {
        dft_prime<R, INV>(v);
    } else if constexpr (R == 6) {
        dft_coprime<2, 3, INV>(v);
    } else if constexpr (R == 10) {
        dft_coprime<2, 5, INV>(v);
    } else if constexpr (R == 9) {
        // 3 x 3 with the twiddles w^1, w^2, w^4, w = e^(-2 pi i / 9)
        using F = decltype(v[0].x);
        T2 a[3][3];
#pragma unroll
        for (int n2 = 0; n2 < 3; ++n2) {
#pragma unroll
            for (int n1 = 0; n1 < 3; ++n1) a[n2][n1] = v[3 * n1 + n2];
            dft_small<3, INV>(a[n2]);
        }
        a[1][1] = rotate<INV>(a[1][1], F(0.7660444431189780352), F(0.64278760968653932632));
        a[1][2] = rotate<INV>(a[1][2], F(0.17364817766693034885), F(0.98480775301220805937));
        a[2][1] = rotate<INV>(a[2][1], F(0.17364817766693034885), F(0.98480775301220805937));
        a[2][2] = rotate<INV>(a[2][2], F(-0.93969262078590838405), F(0.34202014332566873304));
#pragma unroll
        for (int k1 = 0; k1 < 3; ++k1) {
            T2 b[3] = {a[0][k1], a[1][k1], a[2][k1]};
            dft_small<3, INV>(b);
#pragma unroll
            for (int k2 = 0; k2 < 3; ++k2) v[k1 + 3 * k2] = b[k2];
        }
    } else if constexpr (R == 16) {
        // 16 = 4 x 4: inputs x[4 n1 + n2]; a length-4 DFT over n1 for each
        // n2 gives A[n2][k1], then A[n2][k1] w^(n2 k1), then a length-4 DFT
        // over n2 for each k1 gives X[k1 + 4 k2]
        using F = decltype(v[0].x);
        const F c1 = F(0.92387953251128675613), s1 = F(0.38268343236508977173);
        const F c2 = F(0.70710678118654752440);
        T2 a[4][4];
#pragma unroll
        for (int n2 = 0; n2 < 4; ++n2) {
#pragma unroll
            for (int n1 = 0; n1 < 4; ++n1) a[n2][n1] = v[4 * n1 + n2];
            dft_small<4, INV>(a[n2]);
        }
        a[1][1] = rotate<INV>(a[1][1], c1, s1);   // w^1
        a[1][2] = rotate<INV>(a[1][2], c2, c2);   // w^2
        a[1][3] = rotate<INV>(a[1][3], s1, c1);   // w^3
        a[2][1] = rotate<INV>(a[2][1], c2, c2);   // w^2
        {                                        // w^4 = -i (inverse: +i)
            T2 t = a[2][2];
            if (!INV) { a[2][2].x = t.y;  a[2][2].y = -t.x; }
            else      { a[2][2].x = -t.y; a[2][2].y = t.x; }
        }
        a[2][3] = rotate<INV>(a[2][3], -c2, c2);  // w^6
        a[3][1] = rotate<INV>(a[3][1], s1, c1);   // w^3
        a[3][2] = rotate<INV>(a[3][2], -c2, c2);  // w^6
        a[3][3] = rotate<INV>(a[3][3], -c1, -s1); // w^9
#pragma unroll
        for (int k1 = 0; k1 < 4; ++k1) {
            T2 b[4] = {a[0][k1], a[1][k1], a[2][k1], a[3][k1]};
            dft_small<4, INV>(b);
#pragma unroll
            for (int k2 = 0; k2 < 4; ++k2) v[k1 + 4 * k2] = b[k2];
        }
    } else if constexpr (R == 8) {
        // y_k = E_(k mod 4) + w8^k O_(k mod 4), E/O = DFT4 of the even/odd
        // inputs, w8 = e^(-i pi/4) (inverse: conjugate), w8^(k+4) = -w8^k
        T2 e[4] = {v[0], v[2], v[4], v[6]};
        T2 o[4] = {v[1], v[3], v[5], v[7]};
        dft_small<4, INV>(e);
        dft_small<4, INV>(o);
        using F = decltype(v[0].x);
        const F c = F(0.70710678118654752440);
        T2 t1, t2, t3;
        if (!INV) {
            t1.x = (o[1].x + o[1].y) * c; t1.y = (o[1].y - o[1].x) * c;  // (1 - i) c
            t2.x = o[2].y;                t2.y = -o[2].x;                // -i
            t3.x = (o[3].y - o[3].x) * c; t3.y = -(o[3].x + o[3].y) * c; // (-1 - i) c
        } else {
            t1.x = (o[1].x - o[1].y) * c; t1.y = (o[1].x + o[1].y) * c;  // (1 + i) c
            t2.x = -o[2].y;               t2.y = o[2].x;                 // i
            t3.x = -(o[3].x + o[3].y) * c; t3.y = (o[3].x - o[3].y) * c; // (-1 + i) c
        }
        v[0].x = e[0].x + o[0].x; v[0].y = e[0].y + o[0].y;
        v[4].x = e[0].x - o[0].x; v[4].y = e[0].y - o[0].y;
        v[1].x = e[1].x + t1.x;   v[1].y = e[1].y + t1.y;
        v[5].x = e[1].x - t1.x;   v[5].y = e[1].y - t1.y;
        v[2].x = e[2].x + t2.x;   v[2].y = e[2].y + t2.y;
        v[6].x = e[2].x - t2.x;   v[6].y = e[2].y - t2.y;
        v[3].x = e[3].x + t3.x;   v[3].y = e[3].y + t3.y;
        v[7].x = e[3].x - t3.x;   v[7].y = e[3].y - t3.y;
    } else if constexpr (R == 2) {
        T2 a = v[0], b = v[1];
        v[0].x = a.x + b.x; v[0].y = a.y + b.y;
        v[1].x = a.x - b.x; v[1].y = a.y - b.y;
    } else {
        T2 a, b, c, d;
        a.x = v[0].x + v[2].x; a.y = v[0].y + v[2].y;
        b.x = v[0].x - v[2].x; b.y = v[0].y - v[2].y;
        c.x = v[1].x + v[3].x; c.y = v[1].y + v[3].y;
        d.x = v[1].x - v[3].x; d.y = v[1].y - v[3].y;
        v[0].x = a.x + c.x; v[0].y = a.y + c.y;
        v[2].x = a.x - c.x; v[2].y = a.y - c.y;
        if (!INV) {  // y1 = b - i d, y3 = b + i d
            v[1].x = b.x + d.y; v[1].y = b.y - d.x;
            v[3].x = b.x - d.y; v[3].y = b.y + d.x;
        } else {     // y1 = b + i d, y3 = b - i d
            v[1].x = b.x - d.y; v[1].y = b.y + d.x;
            v[3].x = b.x + d.y; v[3].y = b.y - d.x;
        }
    }
}

}  // namespace sc3d
