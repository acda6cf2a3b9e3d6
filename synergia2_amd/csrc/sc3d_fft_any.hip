// sc3d_fft_any.hip -- the Hockney convolution passes for the transform lengths
// the tuned passes of sc3d_fft.hip do not take (those: powers of two, rows of
// gx <= 256 and columns of Dy, Dz <= 512): any length up to 1024, as the
// reference's FFTW plans take any shape (distributed_fft3d_fftw.cc:67-71).
//
// Same inputs, outputs and intermediate layouts as the tuned passes, so the
// two kinds mix per axis (a 48x64x128 grid runs these x passes and the tuned
// y and z passes).  The 1-D transforms are Stockham passes over lines held in
// LDS; a thread computes whole butterflies of a pass in registers (the radix
// selects the code, uniformly over the block).
//
// FP64: the plan splits the length into as few radices of 2..10, 11 and 13 as
// possible; twiddles, then a short DFT (sc3d_dft.h).  Real data are packed in
// pairs: two rows (or two real-even columns of the Green's spectrum) are the
// real and imaginary parts of one complex line.
//
// FP32: factors 4, then primes ascending; every output of a butterfly is the
// sum over its R inputs in order, twiddle and DFT in one table entry per term
// (two consecutive factors run on the elements of one thread where their
// product is a radix below), and rows are transformed one by one.  That is more arithmetic, kept because
// the single-precision field is defined by it to the last bit: another
// factorisation moves the field by 1.4e-7 (rel-L2, as far as either is from
// FP64), which adds up over tracked steps, where runs of one factorisation
// differ by the order of the deposit's atomics alone.
//
// A larger prime factor takes one output per thread, a sum over its R inputs.
//
// What bounds these passes is instruction issue (about 60 % VALU at 20-30
// instructions per element and pass) and the latency of LDS exchanges and
// barriers at the occupancy that the line buffers leave, not bytes.  Measured
// against one output per thread for every factor (R LDS reads and R global
// twiddle reads per output, real rows as full complex lines), us per launch:
//   60x54x100 FP64:  x 26.4 / 27.7 -> 10.8 / 9.7, y 26.3 / 27.4 -> 10.9 / 12.9,
//     z 70.9 -> 18.3, Green's x, y, z 36.8, 25.3, 29.0 -> 17.1, 9.5, 9.8
//   96x80x150 FP32:  x 41.8 -> 13.3, y 42.6 -> 11.1, z' 220 -> 99, y' 114 -> 30,
//     x' 116 -> 35, Green's 64.5, 42.7, 54.5 -> 25.8, 7.9, 14.6
#include <algorithm>
#include <type_traits>
#include <vector>

#include "sc3d_dft.h"
#include "sc3d_green.h"
#include "sc3d_internal.h"

namespace sc3d {

namespace {

constexpr int kAnyThreads = 1024;     // most threads of a block
constexpr int kAnyPreferred = 512;    // ... where it holds several lines per group

// How a block holds its lines: `lines` = groups x per group of (odd) stride
// `st`, tpl threads each.  One line buffer where every pass has a register
// butterfly (all inputs of a pass are read before an output is written), two
// in turn otherwise.
struct AnyShape {
    AnyPlan pl;
    int nl;       // lines (pairs of rows / columns) of one group
    int lines;    // nl * groups
    int st;
    int tpl;
    int two;      // second line buffer
};

// ceil(2^32 / d): n / d = umulhi(n, magic) for n * d < 2^32, d >= 2
inline uint32_t div_magic(uint32_t d) { return uint32_t(((uint64_t(1) << 32) + d - 1) / d); }

// This thread's place in the transforms: its line (< 0: none) and its lane of
// the line.  Neighbouring threads are on neighbouring lines: the odd stride
// keeps them on different banks in every pass, and a column's global accesses
// run across the lines.
struct AnyLane {
    int line, j;
};
__device__ __forceinline__ AnyLane any_lane(const AnyShape& a)
{
    AnyLane q;
    q.j = int(threadIdx.x) / a.lines;
    q.line = int(threadIdx.x) - q.j * a.lines;
    if (q.j >= a.tpl) q.line = -1;
    return q;
}
// The place for loading and storing rows: neighbouring threads along the row.
__device__ __forceinline__ AnyLane any_row_lane(const AnyShape& a)
{
    AnyLane q;
    q.line = int(threadIdx.x) / a.tpl;
    q.j = int(threadIdx.x) - q.line * a.tpl;
    if (q.line >= a.lines) q.line = -1;
    return q;
}

// FP32 takes table butterflies, unpaired rows (see above).
template <typename T2> constexpr bool any_table() { return sizeof(T2) < 16; }

// Butterflies of radix r of one thread in a pass: about ten elements held (four
// wavefronts per SIMD; three radix-4 or radix-5 table butterflies spill).
constexpr int any_per(int r) { return r <= 3 ? 3 : (r <= 5 ? 2 : 1); }
// Radices with a register butterfly (FP64 2..11 and 13, FP32 2..10, 12 and 16;
// 14 and 15 as well spilled, and the scratch slowed every radix: 96x80x150 526
// -> 596 us a step); larger primes (FP32: from 11) go one output per thread.
// Table butterflies of a composite radix are two consecutive passes,
// any_split(r) then r / any_split(r), on the elements of one thread.
constexpr int any_split(int r)
{
    return r == 8 || r == 12 || r == 16 ? 4 : (r == 6 || r == 10 ? 2 : (r == 9 ? 3 : r));
}
constexpr bool any_radix(int r, bool table)
{
    return table ? r <= 10 || r == 12 || r == 16 : r <= 11 || r == 13;
}

// f(radix as a compile-time constant) for the radices of any_radix
template <typename T2, typename F> __device__ __forceinline__ void with_radix(int R, F&& f)
{
    switch (R) {
#define SC3D_ANY_RADIX(r)                                                                      \
    case r:                                                                                    \
        if constexpr (any_radix(r, any_table<T2>())) f(std::integral_constant<int, r>{});      \
        break;
        SC3D_ANY_RADIX(2)
        SC3D_ANY_RADIX(3)
        SC3D_ANY_RADIX(4)
        SC3D_ANY_RADIX(5)
        SC3D_ANY_RADIX(6)
        SC3D_ANY_RADIX(7)
        SC3D_ANY_RADIX(8)
        SC3D_ANY_RADIX(9)
        SC3D_ANY_RADIX(10)
        SC3D_ANY_RADIX(11)
        SC3D_ANY_RADIX(12)
        SC3D_ANY_RADIX(13)
        SC3D_ANY_RADIX(16)
#undef SC3D_ANY_RADIX
    }
}

// A butterfly: outputs X_r = sum_t v_t w_L^(t (ks + r L/N)), ks = k L/(Ns N);
// first: Ns = 1, so ks = 0.
template <int N, bool INV, typename T2>
__device__ __forceinline__ void any_butterfly(T2 (&v)[N], const T2* twl, int NB, int ks,
                                              bool first)
{
    if constexpr (any_table<T2>() && any_split(N) != N) {
        constexpr int A = any_split(N), B = N / A;
        // pass A: butterfly q has the inputs q + B t (L/A = B NB apart); pass
        // B: butterfly r has output r of each, k + r Ns in place of k
        T2 w[A][B];
#pragma unroll
        for (int q = 0; q < B; ++q) {
            T2 u[A];
#pragma unroll
            for (int t = 0; t < A; ++t) u[t] = v[q + B * t];
            any_butterfly<A, INV>(u, twl, B * NB, B * ks, first);
#pragma unroll
            for (int r = 0; r < A; ++r) w[r][q] = u[r];
        }
#pragma unroll
        for (int r = 0; r < A; ++r) {
            any_butterfly<B, INV>(w[r], twl, A * NB, ks + r * NB, first && r == 0);
#pragma unroll
            for (int t = 0; t < B; ++t) v[r + A * t] = w[r][t];
        }
    } else if constexpr (any_table<T2>() && (N == 2 || N == 4)) {
        // w_L^(e + L/4) = -i w_L^e holds exactly in the table (every L that 4
        // divides), so the products of the N outputs are the same ones turned
        // by powers of -i: N - 1 products instead of N (N - 1)
        if (!first) {
#pragma unroll
            for (int t = 1; t < N; ++t) {
                const T2 w = twl[t * ks], x = v[t];
                const auto wy = INV ? -w.y : w.y;
                v[t].x = x.x * w.x - x.y * wy;
                v[t].y = x.x * wy + x.y * w.x;
            }
        }
        T2 out[N];
#pragma unroll
        for (int r = 0; r < N; ++r) {
            T2 s = v[0];
#pragma unroll
            for (int t = 1; t < N; ++t) {
                const int m = t * r * (4 / N) % 4, turn = INV ? (4 - m) % 4 : m;
                s.x += turn == 0 ? v[t].x : turn == 1 ? v[t].y : turn == 2 ? -v[t].x : -v[t].y;
                s.y += turn == 0 ? v[t].y : turn == 1 ? -v[t].x : turn == 2 ? -v[t].y : v[t].x;
            }
            out[r] = s;
        }
#pragma unroll
        for (int r = 0; r < N; ++r) v[r] = out[r];
    } else if constexpr (any_table<T2>()) {
        T2 x[N];
#pragma unroll
        for (int t = 0; t < N; ++t) x[t] = v[t];
#pragma unroll
        for (int r = 0; r < N; ++r) {
            T2 s = x[0];
#pragma unroll
            for (int t = 1; t < N; ++t) {
                // t ks < L and (t r mod N) L/N < L: the table holds two periods
                const T2 w = twl[t * ks + (t * r % N) * NB];
                const auto wy = INV ? -w.y : w.y;
                s.x += x[t].x * w.x - x[t].y * wy;
                s.y += x[t].x * wy + x[t].y * w.x;
            }
            v[r] = s;
            // one output's twiddles in flight (all of them spill)
            __builtin_amdgcn_sched_barrier(0);
        }
    } else {
        if (!first) {
#pragma unroll
            for (int r = 1; r < N; ++r) v[r] = twmul<INV>(v[r], twl[r * ks]);
        }
        dft_small<N, INV>(v);
    }
}

// The inputs b + r L/N of butterfly b out of a line, and their butterfly.
template <int N, bool INV, typename T2>
__device__ __forceinline__ void any_read(T2 (&v)[N], const T2* lb, const T2* twl, int b, int NB,
                                         int Ns, int k)
{
#pragma unroll
    for (int r = 0; r < N; ++r) v[r] = lb[b + r * NB];
    any_butterfly<N, INV>(v, twl, NB, k * (NB / Ns), Ns == 1);
}

// Radix R without a register butterfly: output (j/Ns)*Ns*R + j%Ns + r*Ns is
// sum_t x[j + t L/R] w_L^(t (k L/(Ns R) + r L/R)), k = j % Ns -- twiddle and
// length-R DFT in one table lookup per term.  out(p, value) takes the outputs.
template <bool INV, typename T2, typename Out>
__device__ __forceinline__ void any_direct(const AnyShape& a, const AnyLane& q, const T2* src,
                                           const T2* twl, int R, int Ns, uint32_t magic,
                                           Out&& out)
{
    using F = decltype(T2{}.x);
    if (q.line < 0) return;
    const int L = a.pl.L, LR = L / R, tstep = LR / Ns;
    const T2* lb = src + q.line * a.st;
    for (int o = q.j; o < L; o += a.tpl) {
        const int rest = Ns > 1 ? int(__umulhi(uint32_t(o), magic)) : o, k = o - rest * Ns;
        const int jb = rest / R, r = rest - jb * R;
        const int base = k * tstep + r * LR;  // < L
        F ax = F(0), ay = F(0);
        int e = 0;
        for (int t = 0, at = jb * Ns + k; t < R; ++t, at += LR) {
            const T2 x = lb[at];
            const T2 w = twl[e];
            const F wy = INV ? -w.y : w.y;
            ax += x.x * w.x - x.y * wy;
            ay += x.x * wy + x.y * w.x;
            e += base;
            if (e >= L) e -= L;
        }
        T2 s;
        s.x = ax;
        s.y = ay;
        out(o, s);
    }
}

// A pass between line buffers: radix R after the radices whose product is Ns.
// Synchronised on return; src and dst change places where there are two.
template <bool INV, typename T2>
__device__ __forceinline__ void any_mid(const AnyShape& a, const AnyLane& q, T2*& buf, T2*& alt,
                                        const T2* twl, int R, int Ns, uint32_t magic)
{
    T2* dst = a.two ? alt : buf;
    if (!any_radix(R, any_table<T2>())) {
        any_direct<INV>(a, q, buf, twl, R, Ns, magic,
                        [&](int p, T2 s) { dst[q.line * a.st + p] = s; });
    } else {
        with_radix<T2>(R, [&](auto rc) {
            constexpr int N = decltype(rc)::value, Q = any_per(N);
            const int NB = a.pl.L / N;
            T2 v[Q][N];
            int d[Q];
#pragma unroll
            for (int u = 0; u < Q; ++u) {
                const int at = q.j + u * a.tpl, b = min(at, NB - 1);
                const int blk = Ns > 1 ? int(__umulhi(uint32_t(b), magic)) : b;
                const int k = b - blk * Ns, line = max(q.line, 0);
                any_read<N, INV>(v[u], buf + line * a.st, twl, b, NB, Ns, k);
                d[u] = q.line >= 0 && at < NB ? line * a.st + blk * Ns * N + k : -1;
            }
            if (!a.two) __syncthreads();
#pragma unroll
            for (int u = 0; u < Q; ++u) {
                if (d[u] < 0) continue;
#pragma unroll
                for (int r = 0; r < N; ++r) dst[d[u] + r * Ns] = v[u][r];
            }
        });
    }
    __syncthreads();
    if (a.two) {
        alt = buf;
        buf = dst;
    }
}

// The first pass from io.load (the inputs b + r NB of butterfly b) into `buf`
// (no other pass may be reading it); synchronised on return (the twiddles
// too).
template <bool INV, typename T2, typename IO>
__device__ __forceinline__ void any_first(const AnyShape& a, const AnyLane& q, T2* buf,
                                          const T2* twl, const IO& io)
{
    if constexpr (any_table<T2>()) __syncthreads();  // the twiddles
    if (q.line >= 0) with_radix<T2>(a.pl.R[0], [&](auto rc) {
        constexpr int N = decltype(rc)::value, Q = any_per(N);
        const int NB = a.pl.L / N;
        T2 v[Q][N];
#pragma unroll
        for (int u = 0; u < Q; ++u) io.load(min(q.j + u * a.tpl, NB - 1), NB, v[u]);
#pragma unroll
        for (int u = 0; u < Q; ++u) {
            const int b = q.j + u * a.tpl;
            any_butterfly<N, INV>(v[u], twl, NB, 0, true);
            if (b >= NB) continue;
            T2* lb = buf + q.line * a.st + b * N;
#pragma unroll
            for (int r = 0; r < N; ++r) lb[r] = v[u][r];
        }
    });
    __syncthreads();
}

// The last pass (radix R, Ns = L / R) out of `buf` into io.store (the outputs
// b + r NB of butterfly b; store1: one element).
template <bool INV, typename T2, typename IO>
__device__ __forceinline__ void any_last(const AnyShape& a, const AnyLane& q, const T2* buf,
                                         const T2* twl, int R, uint32_t magic, const IO& io)
{
    if (!any_radix(R, any_table<T2>())) {
        any_direct<INV>(a, q, buf, twl, R, a.pl.L / R, magic,
                        [&](int p, T2 v) { io.store1(p, v); });
        return;
    }
    with_radix<T2>(R, [&](auto rc) {
        constexpr int N = decltype(rc)::value, Q = any_per(N);
        const int NB = a.pl.L / N;
#pragma unroll
        for (int u = 0; u < Q; ++u) {
            const int b = q.j + u * a.tpl;
            if (q.line < 0 || b >= NB) continue;
            T2 v[N];
            any_read<N, INV>(v, buf + q.line * a.st, twl, b, NB, NB, b);
            io.store(b, NB, v);
        }
    });
}

// A whole transform of columns.
template <bool INV, typename T2, typename IO>
__device__ __forceinline__ void any_columns(const AnyShape& a, const AnyLane& q, T2* buf, T2* alt,
                                            const T2* twl, const IO& io)
{
    any_first<INV>(a, q, buf, twl, io);
    int Ns = a.pl.R[0], s = 1;
    for (; s < a.pl.np - 1; ++s) {
        any_mid<INV>(a, q, buf, alt, twl, a.pl.R[s], Ns, a.pl.ns_magic[s]);
        Ns *= a.pl.R[s];
    }
    any_last<INV>(a, q, buf, twl, a.pl.R[s], a.pl.ns_magic[s], io);
}

// The z passes: forward; the spectrum through sp.mul, and for a second group
// (K = 2) that through sp.derive; inverse.  The inverse takes the radices in reverse, so the butterfly that ends
// the forward transform holds the inputs of the one that starts the inverse.
// The forward transform is on the first group's lines (`q` of the others
// idles); K groups of a.nl lines come back.
template <int K, typename T2, typename IO, typename Spectrum>
__device__ __forceinline__ void any_convolve(const AnyShape& a, const AnyLane& q, T2* buf, T2* alt,
                                             const T2* twl, const IO& io, const Spectrum& sp)
{
    AnyLane f = q;
    if (f.line >= a.nl) f.line = -1;
    any_first<false>(a, f, buf, twl, io);
    const int np = a.pl.np;
    int Ns = a.pl.R[0];
    for (int s = 1; s < np - 1; ++s) {
        any_mid<false>(a, f, buf, alt, twl, a.pl.R[s], Ns, a.pl.ns_magic[s]);
        Ns *= a.pl.R[s];
    }
    const int R = a.pl.R[np - 1];
    if constexpr (any_table<T2>()) {
        // the inverse takes the radices in the same order: the spectrum goes
        // back to LDS, each element where its butterfly's thread read it
        T2* dst = buf;
        if (!any_radix(R, true)) {
            dst = alt;
            any_direct<false>(a, f, buf, twl, R, Ns, a.pl.ns_magic[np - 1], [&](int p, T2 u) {
                T2 v[1] = {u};
                sp.mul(p, 0, v);
                dst[f.line * a.st + p] = v[0];
                if constexpr (K == 2) {
                    sp.derive(p, 0, v);
                    dst[(f.line + a.nl) * a.st + p] = v[0];
                }
            });
        } else {
            with_radix<T2>(R, [&](auto rc) {
                constexpr int N = decltype(rc)::value, Q = any_per(N);
                const int NB = a.pl.L / N;
#pragma unroll
                for (int u = 0; u < Q; ++u) {
                    const int b = f.j + u * a.tpl;
                    if (f.line < 0 || b >= NB) continue;
                    T2 v[N];
                    any_read<N, false>(v, buf + f.line * a.st, twl, b, NB, NB, b);
                    sp.mul(b, NB, v);
                    T2* lb = dst + f.line * a.st + b;
#pragma unroll
                    for (int r = 0; r < N; ++r) lb[r * NB] = v[r];
                    if constexpr (K == 2) {
                        sp.derive(b, NB, v);
#pragma unroll
                        for (int r = 0; r < N; ++r) lb[a.nl * a.st + r * NB] = v[r];
                    }
                }
            });
        }
        __syncthreads();
        if (dst != buf) {
            alt = buf;
            buf = dst;
        }
        Ns = 1;
        for (int s = 0; s < np - 1; ++s) {
            any_mid<true>(a, q, buf, alt, twl, a.pl.R[s], Ns, a.pl.ns_magic[s]);
            Ns *= a.pl.R[s];
        }
        any_last<true>(a, q, buf, twl, R, a.pl.ns_magic[np - 1], io);
        return;
    } else {
        T2* dst = a.two ? alt : buf;
        if (!any_radix(R, any_table<T2>())) {
            any_direct<false>(a, f, buf, twl, R, Ns, a.pl.ns_magic[np - 1], [&](int p, T2 u) {
                T2 v[1] = {u};
                sp.mul(p, 0, v);
                dst[f.line * a.st + p] = v[0];
                if constexpr (K == 2) {
                    sp.derive(p, 0, v);
                    dst[(f.line + a.nl) * a.st + p] = v[0];
                }
            });
            __syncthreads();
            alt = buf;  // a direct radix always has the second buffer
            buf = dst;
            any_mid<true>(a, q, buf, alt, twl, R, 1, 0u);
        } else {
            with_radix<T2>(R, [&](auto rc) {
                constexpr int N = decltype(rc)::value, Q = any_per(N);
                const int NB = a.pl.L / N;
                T2 v[Q][N];
#pragma unroll
                for (int u = 0; u < Q; ++u) {
                    const int b = min(f.j + u * a.tpl, NB - 1);
                    any_read<N, false>(v[u], buf + max(f.line, 0) * a.st, twl, b, NB, NB, b);
                }
                if (!a.two) __syncthreads();
#pragma unroll
                for (int u = 0; u < Q; ++u) {
                    const int b = f.j + u * a.tpl;
                    if (f.line < 0 || b >= NB) continue;
                    sp.mul(b, NB, v[u]);
                    T2* lb = dst + f.line * a.st + b * N;
                    if constexpr (K == 2) {
                        T2 w[N];
#pragma unroll
                        for (int r = 0; r < N; ++r) w[r] = v[u][r];
                        sp.derive(b, NB, w);
                        dft_small<N, true>(w);
#pragma unroll
                        for (int r = 0; r < N; ++r) lb[a.nl * a.st + r] = w[r];
                    }
                    dft_small<N, true>(v[u]);
#pragma unroll
                    for (int r = 0; r < N; ++r) lb[r] = v[u][r];
                }
            });
            __syncthreads();
            if (a.two) {
                alt = buf;
                buf = dst;
            }
        }
        Ns = R;
        for (int s = np - 2; s > 0; --s) {
            any_mid<true>(a, q, buf, alt, twl, a.pl.R[s], Ns, a.pl.back_magic[s]);
            Ns *= a.pl.R[s];
        }
        any_last<true>(a, q, buf, twl, a.pl.R[0], a.pl.back_magic[0], io);
    }
}

// The rows in `buf` transformed in LDS; returns the buffer that holds the
// result.  The caller has synchronised after filling buf and the twiddles;
// synchronised on return.
template <bool INV, typename T2>
__device__ __forceinline__ T2* any_rows(const AnyShape& a, T2* buf, T2* alt, const T2* twl)
{
    const AnyLane q = any_lane(a);
    int Ns = 1;
    for (int s = 0; s < a.pl.np; ++s) {
        any_mid<INV>(a, q, buf, alt, twl, a.pl.R[s], Ns, a.pl.ns_magic[s]);
        Ns *= a.pl.R[s];
    }
    return buf;
}

// LDS of a block: the twiddle table (two periods of it for table butterflies),
// the line buffer, the second one.
template <typename T2> constexpr int any_periods() { return any_table<T2>() ? 2 : 1; }
template <typename T2> struct AnyLds {
    T2 *twl, *buf, *alt;
};
template <typename T2>
__device__ __forceinline__ AnyLds<T2> any_lds(const AnyShape& a, const T2* __restrict__ tw)
{
    extern __shared__ __align__(16) unsigned char any_smem[];
    AnyLds<T2> m;
    m.twl = reinterpret_cast<T2*>(any_smem);
    m.buf = m.twl + any_periods<T2>() * a.pl.L;
    m.alt = m.buf + a.lines * a.st;
    for (int e = threadIdx.x; e < a.pl.L; e += blockDim.x) {
        m.twl[e] = tw[e];
        if constexpr (any_table<T2>()) m.twl[a.pl.L + e] = tw[e];
    }
    return m;
}

// Column groups in an XCD-contiguous order (neighbouring groups share
// 128-byte lines of S); grids are multiples of 8.
__device__ __forceinline__ int any_group()
{
    return int(blockIdx.x & 7u) * int(gridDim.x >> 3) + int(blockIdx.x >> 3);
}

template <typename T2, typename R>
__device__ __forceinline__ T2 times_minus_i(T2 v, R s)  // v * (-i s)
{
    T2 o;
    o.x = s * v.y;
    o.y = -(s * v.x);
    return o;
}

// sin(2 pi k / L) = -Im of the length-L table's entry k (exactly 0 at k = 0
// and k = L/2).
template <typename T2> __device__ __forceinline__ auto any_sin(const T2* tw, int k)
{
    return -tw[k].y;
}

template <typename T2> __device__ __forceinline__ T2 czero()
{
    T2 v;
    v.x = decltype(v.x)(0);
    v.y = decltype(v.x)(0);
    return v;
}

// Rows (or real-even columns) of one line.
template <typename T2> constexpr int any_rows_per() { return any_table<T2>() ? 1 : 2; }

// The spectra of a line's rows out of Z[k] and Z[L-k]: rows A and B are
// Z = A + i B; one row is Z itself.
template <typename T2>
__device__ __forceinline__ void unpack_pair(T2 zk, T2 zm, T2& A, T2& B)
{
    using F = decltype(zk.x);
    if constexpr (any_rows_per<T2>() == 1) {
        A = zk;
    } else {
        A.x = F(0.5) * (zk.x + zm.x);
        A.y = F(0.5) * (zk.y - zm.y);
        B.x = F(0.5) * (zk.y + zm.y);
        B.y = F(0.5) * (zm.x - zk.x);
    }
}
// ... and of Hermitian rows into Z[k] and Z[L-k]:
template <typename T2>
__device__ __forceinline__ void pack_pair(T2 A, T2 B, T2& zk, T2& zm)
{
    if constexpr (any_rows_per<T2>() == 1) {
        zk = A;
        zm.x = A.x;
        zm.y = -A.y;
    } else {
        zk.x = A.x - B.y;
        zk.y = A.y + B.x;
        zm.x = A.x + B.y;
        zm.y = B.x - A.y;
    }
}

// A column's elements p at col[p * ps].  HALF_IN: those from L/2 on are zero
// and not read.  HALF_OUT: those are not stored.  Radix N, r: element
// b + r L/N, so for the even N the halves are whole values of r, for an odd N
// r = (N-1)/2 straddles the middle; no other element needs a condition (which
// costs a branch each, and the loads of a butterfly leave one at a time: y'
// pass of 96x80x150 FP32 48 -> 27 us without).  A line that does not exist reads line 0
// of its job and stores nothing.
template <typename T2, bool HALF_IN, bool HALF_OUT> struct AnyColumn {
    T2* col;
    int ps, half;
    bool live;
    template <int N> __device__ __forceinline__ void load(int b, int NB, T2 (&v)[N]) const
    {
#pragma unroll
        for (int r = 0; r < N; ++r) {
            const int p = b + r * NB;
            if (!HALF_IN || 2 * r + 1 < N) {
                v[r] = col[p * ps];
            } else if (2 * r + 1 == N) {
                const T2 x = col[min(p, half - 1) * ps];
                v[r].x = p < half ? x.x : decltype(x.x)(0);
                v[r].y = p < half ? x.y : decltype(x.x)(0);
            } else {
                v[r] = czero<T2>();
            }
        }
    }
    template <int N> __device__ __forceinline__ void store(int b, int NB, T2 (&v)[N]) const
    {
        if (!live) return;
#pragma unroll
        for (int r = 0; r < N; ++r) {
            const int p = b + r * NB;
            if (!HALF_OUT || 2 * r + 1 < N || (2 * r + 1 == N && p < half)) col[p * ps] = v[r];
        }
    }
    __device__ __forceinline__ void store1(int p, T2 v) const
    {
        if (live && (!HALF_OUT || p < half)) col[p * ps] = v;
    }
};

// The Green's spectrum (and the correction spectrum chat, where the shape has
// one) on a column; derive: times D_z = -i sin(2 pi p / L) / h_z.
template <typename T2, typename R> struct AnySpectrum {
    const R* g;
    const T2* c;
    int gs, cs, L;
    const T2* twl;
    R ihz;
    template <int N> __device__ __forceinline__ void mul(int b, int NB, T2 (&v)[N]) const
    {
        R gv[N];
#pragma unroll
        for (int r = 0; r < N; ++r) {
            const int p = b + r * NB;
            gv[r] = g[min(p, L - p) * gs];
        }
        if (c) {
#pragma unroll
            for (int r = 0; r < N; ++r) {
                const T2 u = v[r], e = c[(b + r * NB) * cs];
                v[r].x = u.x * gv[r] + (u.x * e.x - u.y * e.y);
                v[r].y = u.y * gv[r] + (u.x * e.y + u.y * e.x);
            }
        } else {
#pragma unroll
            for (int r = 0; r < N; ++r) {
                v[r].x *= gv[r];
                v[r].y *= gv[r];
            }
        }
    }
    template <int N> __device__ __forceinline__ void derive(int b, int NB, T2 (&v)[N]) const
    {
#pragma unroll
        for (int r = 0; r < N; ++r) v[r] = times_minus_i(v[r], any_sin(twl, b + r * NB) * ihz);
    }
};

}  // namespace

// ---------------------------------------------------------------------------
// x pass, forward.  FULL false: rho rows (z < gz, y < gy; gx
// reals, zero to Dx) -> S rows kx = 0..gx.  Precision form: unit-peak scaling
// on load, as the tuned pass.  FULL: rows of Dx reals of C -> rows of chat,
// where h changed (the g2 correction).
// ---------------------------------------------------------------------------
template <typename R, bool FULL>
__global__ __launch_bounds__(kAnyThreads, 4) void ga_x_r2c(
    const GridJob* __restrict__ jobs, const typename cplx<R>::type* __restrict__ tw, AnyShape a,
    int nrows, int gx, int gy, int Dy, const R* __restrict__ C,
    typename cplx<R>::type* __restrict__ chat)
{
    using T2 = typename cplx<R>::type;
    const GridJob& J = jobs[blockIdx.y];
    const R* __restrict__ in = FULL ? C : in_memory(static_cast<const R*>(J.rho));
    T2* __restrict__ S = FULL ? chat : in_memory(static_cast<T2*>(J.S));
    const DomainRec* dom = in_memory(J.dom);
    if (dom->error || (FULL && !dom->ghat_dirty)) return;
    AnyLds<T2> m = any_lds(a, tw);
    const AnyLane q = any_row_lane(a);
    const int L = a.pl.L, Hx = gx + 1, nin = FULL ? L : gx;
    constexpr int W = any_rows_per<T2>();
    const int r0 = W * (int(blockIdx.x) * a.nl + q.line), r1 = W == 2 ? r0 + 1 : nrows;
    const float peak = __int_as_float(dom->rho_peak);
    const bool unit_peak = !FULL && sizeof(R) == sizeof(float) && peak > 0.0f;
    if (q.line >= 0)
        for (int x = q.j; x < L; x += a.tpl) {
            T2 v = czero<T2>();
            if (x < nin) {
                if (r0 < nrows) v.x = in[int64_t(r0) * nin + x];
                if (r1 < nrows) v.y = in[int64_t(r1) * nin + x];
                if (unit_peak) {
                    v.x = R(v.x / peak);
                    v.y = R(v.y / peak);
                }
            }
            m.buf[q.line * a.st + x] = v;
        }
    __syncthreads();
    const T2* out = any_rows<false>(a, m.buf, m.alt, m.twl);
    if (q.line < 0 || r0 >= nrows) return;
    auto row = [&](int r) -> int64_t {
        if (FULL) return int64_t(r) * Hx;
        const int z = r / gy, y = r - z * gy;
        return (int64_t(z) * Dy + y) * Hx;
    };
    T2* s0 = S + row(r0);
    T2* s1 = S + (r1 < nrows ? row(r1) : 0);
    const T2* lb = out + q.line * a.st;
    for (int k = q.j; k < Hx; k += a.tpl) {
        T2 A, B;
        unpack_pair(lb[k], lb[k == 0 ? 0 : L - k], A, B);
        s0[k] = A;
        if (r1 < nrows) s1[k] = B;
    }
}

// x pass, inverse (C2R): S rows -> potential rows x < gx.  The
// imaginary parts of the DC and Nyquist terms are ignored (FFTW c2r).
template <typename R>
__global__ __launch_bounds__(kAnyThreads, 4) void ga_x_c2r(
    const GridJob* __restrict__ jobs, const typename cplx<R>::type* __restrict__ tw, AnyShape a,
    int nrows, int gx, int gy, int Dy)
{
    using T2 = typename cplx<R>::type;
    const GridJob& J = jobs[blockIdx.y];
    const T2* __restrict__ S = in_memory(static_cast<const T2*>(J.S));
    R* __restrict__ phi = in_memory(static_cast<R*>(J.phi));
    const DomainRec* dom = in_memory(J.dom);
    if (dom->error) return;
    AnyLds<T2> m = any_lds(a, tw);
    const AnyLane q = any_row_lane(a);
    const int L = a.pl.L, Hx = gx + 1;
    constexpr int W = any_rows_per<T2>();
    const int r0 = W * (int(blockIdx.x) * a.nl + q.line), r1 = W == 2 ? r0 + 1 : nrows;
    auto row = [&](int r) {
        const int z = r / gy, y = r - z * gy;
        return S + (int64_t(z) * Dy + y) * Hx;
    };
    if (q.line >= 0) {
        T2* lb = m.buf + q.line * a.st;
        const T2* s0 = row(r0 < nrows ? r0 : 0);
        const T2* s1 = row(r1 < nrows ? r1 : 0);
        for (int k = q.j; k < Hx; k += a.tpl) {
            T2 A = czero<T2>(), B = A, zk, zm;
            if (r0 < nrows) A = s0[k];
            if (r1 < nrows) B = s1[k];
            if (k == 0 || k == gx) A.y = B.y = R(0);
            pack_pair(A, B, zk, zm);
            lb[k] = zk;
            if (k > 0 && k < gx) lb[L - k] = zm;
        }
    }
    __syncthreads();
    const T2* out = any_rows<true>(a, m.buf, m.alt, m.twl);
    if (q.line < 0) return;
    const T2* lb = out + q.line * a.st;
    for (int x = q.j; x < gx; x += a.tpl) {
        const T2 v = lb[x];
        if (r0 < nrows) phi[int64_t(r0) * gx + x] = v.x;
        if (r1 < nrows) phi[int64_t(r1) * gx + x] = v.y;
    }
}

// Column passes over S, as k_cols_reg: line l -> (plane = l / lpp, c = l % lpp),
// element p at S[plane*plane_stride + p*pstride + c].  MODE 0 forward from the
// non-zero half, 1 inverse keeping the half, 2 forward x Green's spectrum,
// inverse (the z pass), half in and out, 3 forward of whole columns of `over`
// where h changed (the g2 correction spectrum, any_chat).
template <typename R, int MODE>
__global__ __launch_bounds__(kAnyThreads, 4) void ga_cols(
    const GridJob* __restrict__ jobs, const typename cplx<R>::type* __restrict__ tw, AnyShape a,
    int nlines, int lpp, int plane_stride, int pstride, int gy, int Hx,
    typename cplx<R>::type* over)
{
    using T2 = typename cplx<R>::type;
    const GridJob& J = jobs[blockIdx.y];
    T2* __restrict__ S = MODE == 3 ? over : in_memory(static_cast<T2*>(J.S));
    const DomainRec* dom = in_memory(J.dom);
    if (dom->error || (MODE == 3 && !dom->ghat_dirty)) return;
    AnyLds<T2> m = any_lds(a, tw);
    const AnyLane q = any_lane(a);
    const int L = a.pl.L;
    int l = any_group() * a.nl + q.line;
    const bool live = q.line >= 0 && l < nlines;
    if (!live) l = 0;
    const int plane = l / lpp;
    AnyColumn<T2, MODE == 0 || MODE == 2, MODE == 1 || MODE == 2> io;
    io.col = S + int64_t(plane) * plane_stride + (l - plane * lpp);
    io.ps = pstride;
    io.half = L / 2;
    io.live = live;
    if constexpr (MODE == 2) {
        const int Dy = lpp / Hx;
        const int ky = l / Hx, kx = l - ky * Hx;
        const R* ghat = in_memory(static_cast<const R*>(J.ghat));
        const T2* chat = in_memory(static_cast<const T2*>(J.chat));
        const AnySpectrum<T2, R> sp{ghat + min(ky, Dy - ky) * Hx + kx, chat ? chat + l : nullptr,
                                    (gy + 1) * Hx, lpp, L, m.twl, R(0)};
        any_convolve<1>(a, q, m.buf, m.alt, m.twl, io, sp);
    } else {
        any_columns<MODE == 1>(a, q, m.buf, m.alt, m.twl, io);
    }
}

// ---------------------------------------------------------------------------
// Precision form: the field straight from the spectrum, as k_z_field_reg /
// k_y_field_reg / k_x_field (D_a(k) = -i sin(2 pi k / D_a) / h_a).
// z : per (ky, kx) column: forward, x Ghat, inverse of T and of T*D_z,
//     keep z < gz: T -> S, T_z -> S2
// The lines of the second group are idle in the forward transform.
// ---------------------------------------------------------------------------
template <typename R>
__global__ __launch_bounds__(kAnyThreads, 4) void ga_z_field(
    const GridJob* __restrict__ jobs, const typename cplx<R>::type* __restrict__ tw, AnyShape a,
    int nlines, int gy, int Hx)
{
    using T2 = typename cplx<R>::type;
    const GridJob& J = jobs[blockIdx.y];
    const R* __restrict__ ghat = in_memory(static_cast<const R*>(J.ghat));
    const T2* __restrict__ chat = in_memory(static_cast<const T2*>(J.chat));
    const DomainRec* dom = in_memory(J.dom);
    if (dom->error) return;
    AnyLds<T2> m = any_lds(a, tw);
    const AnyLane q = any_lane(a);
    const bool second = q.line >= a.nl;
    const int L = a.pl.L, Dy = nlines / Hx;
    int l = any_group() * a.nl + (second ? q.line - a.nl : q.line);
    const bool live = q.line >= 0 && l < nlines;
    if (!live) l = 0;
    const int ky = l / Hx, kx = l - ky * Hx;
    const AnyColumn<T2, true, true> io{in_memory(static_cast<T2*>(second ? J.S2 : J.S)) + l, nlines,
                                       L / 2, live};
    const AnySpectrum<T2, R> sp{ghat + min(ky, Dy - ky) * Hx + kx, chat ? chat + l : nullptr,
                                (gy + 1) * Hx, nlines, L, m.twl, R(dom->inv_h[2])};
    any_convolve<2>(a, q, m.buf, m.alt, m.twl, io, sp);
}

// y': per (z < gz, kx) column: inverse of T, T*D_y and T_z, keep y < gy:
// S rows [0, gy) <- T, S rows [gy, Dy) <- T*D_y, S2 rows [0, gy) <- T_z.  The
// groups of T and T*D_y both read the column: every load comes before the
// barrier that ends the first pass, every store after it.
template <typename T2, typename R> struct AnyFieldColumn : AnyColumn<T2, false, true> {
    const T2* in;
    const T2* twl;
    R ihy;
    bool derive;
    template <int N> __device__ __forceinline__ void load(int b, int NB, T2 (&v)[N]) const
    {
#pragma unroll
        for (int r = 0; r < N; ++r) {
            const T2 x = in[(b + r * NB) * this->ps];
            const T2 d = times_minus_i(x, any_sin(twl, b + r * NB) * ihy);
            v[r].x = derive ? d.x : x.x;
            v[r].y = derive ? d.y : x.y;
        }
    }
};

template <typename R>
__global__ __launch_bounds__(kAnyThreads, 4) void ga_y_field(
    const GridJob* __restrict__ jobs, const typename cplx<R>::type* __restrict__ tw, AnyShape a,
    int nlines, int gy, int Hx)
{
    using T2 = typename cplx<R>::type;
    const GridJob& J = jobs[blockIdx.y];
    const DomainRec* dom = in_memory(J.dom);
    if (dom->error) return;
    AnyLds<T2> m = any_lds(a, tw);
    const AnyLane q = any_lane(a);
    const int f = max(q.line, 0) / a.nl;  // T, T*D_y, T_z
    const int L = a.pl.L;
    int l = any_group() * a.nl + (q.line - f * a.nl);
    const bool live = q.line >= 0 && l < nlines;
    if (!live) l = 0;
    const int z = l / Hx;
    AnyFieldColumn<T2, R> io;
    T2* in = in_memory(static_cast<T2*>(f == 2 ? J.S2 : J.S)) + int64_t(z) * L * Hx + (l - z * Hx);
    io.col = in + (f == 1 ? gy * Hx : 0);
    io.ps = Hx;
    io.half = gy;
    io.live = live;
    io.in = in;
    io.twl = m.twl;
    io.ihy = R(dom->inv_h[1]);
    io.derive = f == 1;
    __syncthreads();  // the twiddles
    any_columns<true>(a, q, m.buf, m.alt, m.twl, io);
}

// x': per row (z < gz, y < gy): C2R of (S row) * D_x, of S row
// gy + y and of the S2 row -> E (x, y, z, 0) on interior nodes, 0 on the
// boundary.  gx_magic: division by gx.
template <typename R>
__global__ __launch_bounds__(kAnyThreads, 4) void ga_x_field(
    const GridJob* __restrict__ jobs, const typename cplx<R>::type* __restrict__ tw, AnyShape a,
    int gx, int gy, int gz, int Dy, uint32_t gx_magic)
{
    using T2 = typename cplx<R>::type;
    using T4 = typename vec4_of<R>::type;
    const GridJob& J = jobs[blockIdx.y];
    const T2* __restrict__ S = in_memory(static_cast<const T2*>(J.S));
    const T2* __restrict__ S2 = in_memory(static_cast<const T2*>(J.S2));
    T4* __restrict__ E = in_memory(static_cast<T4*>(J.E));
    const DomainRec* dom = in_memory(J.dom);
    if (dom->error) return;
    AnyLds<T2> m = any_lds(a, tw);
    const AnyLane q = any_row_lane(a);
    const int f = q.line < 0 ? 0 : q.line / a.nl;
    const R ihx = R(dom->inv_h[0]);
    const int L = a.pl.L, Hx = gx + 1;
    const int nrows = gz * gy;
    constexpr int W = any_rows_per<T2>();
    const int first = W * int(blockIdx.x) * a.nl;
    if (q.line >= 0) {
        const int r0 = first + W * (q.line - f * a.nl), r1 = W == 2 ? r0 + 1 : nrows;
        auto row = [&](int r) {
            const int z = r / gy, y = r - z * gy;
            return (f == 2 ? S2 : S) + (int64_t(z) * Dy + y + (f == 1 ? gy : 0)) * Hx;
        };
        const T2* s0 = row(r0 < nrows ? r0 : 0);
        const T2* s1 = row(r1 < nrows ? r1 : 0);
        T2* lb = m.buf + q.line * a.st;
        for (int k = q.j; k < Hx; k += a.tpl) {
            T2 A = czero<T2>(), B = A, zk, zm;
            if (r0 < nrows) A = s0[k];
            if (r1 < nrows) B = s1[k];
            if (k == 0 || k == gx) A.y = B.y = R(0);
            if (f == 0) {
                const R d = any_sin(tw, k) * ihx;
                A = times_minus_i(A, d);
                B = times_minus_i(B, d);
            }
            pack_pair(A, B, zk, zm);
            lb[k] = zk;
            if (k > 0 && k < gx) lb[L - k] = zm;
        }
    }
    __syncthreads();
    const T2* out = any_rows<true>(a, m.buf, m.alt, m.twl);
    for (int e = threadIdx.x; e < W * a.nl * gx; e += blockDim.x) {
        const int i = int(__umulhi(uint32_t(e), gx_magic)), x = e - i * gx;
        const int r = first + i;
        if (r >= nrows) break;
        const int z = r / gy, y = r - z * gy;
        T4 o;
        o.x = R(0);
        o.y = R(0);
        o.z = R(0);
        o.w = R(0);
        if (x > 0 && x < gx - 1 && y > 0 && y < gy - 1 && z > 0 && z < gz - 1) {
            const T2* lb = out + i / W * a.st + x;
            const T2 vx = lb[0], vy = lb[a.nl * a.st], vz = lb[2 * a.nl * a.st];
            const bool im = i % W != 0;
            o.x = im ? vx.y : vx.x;
            o.y = im ? vy.y : vy.x;
            o.z = im ? vz.y : vz.x;
        }
        E[int64_t(r) * gx + x] = o;
    }
}

// ---------------------------------------------------------------------------
// Green's spectrum, as k_green_x / k_green_cols: rows (Z <= gz, Y <= gy) of
// the doubled grid generated (FP64 values, rounded once to T) and
// transformed along x, keeping the real kx = 0..gx (the row is even);
// then real-even column transforms along y (AXIS 1) and z (AXIS 2) in place
// over the octant, keeping p <= L/2.  Real-even data transform to real data,
// so a pair comes out as the real and imaginary parts it went in as.
// ---------------------------------------------------------------------------
template <typename T> __device__ __forceinline__ T* any_ghat(const GridJob& J)
{
    return in_memory(sizeof(T) == sizeof(double) ? reinterpret_cast<T*>(J.ghat64)
                                                 : static_cast<T*>(J.ghat));
}

template <typename T>
__global__ __launch_bounds__(kAnyThreads, 4) void ga_green_x(
    const GridJob* __restrict__ jobs, const typename cplx<T>::type* __restrict__ tw, AnyShape a,
    int gx, int gy, int gz, int green_fn)
{
    using T2 = typename cplx<T>::type;
    const GridJob& J = jobs[blockIdx.y];
    T* __restrict__ ghat = any_ghat<T>(J);
    const DomainRec* dom = in_memory(J.dom);
    if (dom->error || !dom->ghat_dirty) return;
    AnyLds<T2> m = any_lds(a, tw);
    const AnyLane q = any_row_lane(a);
    const int L = a.pl.L, Hx = gx + 1;
    const int nrows = (gz + 1) * (gy + 1);
    constexpr int W = any_rows_per<T2>();
    const int r0 = W * (int(blockIdx.x) * a.nl + q.line), r1 = W == 2 ? r0 + 1 : nrows;
    const double hx = dom->h[0], hy = dom->h[1], hz = dom->h[2];
    if (q.line >= 0) {
        T2* lb = m.buf + q.line * a.st;
        auto value = [&](int r, int x) -> T {
            if (r >= nrows) return T(0);
            const int Z = r / (gy + 1), Y = r - Z * (gy + 1);
            return T(green_value(green_fn, x * hx, Y * hy, Z * hz, hx, hy, hz));
        };
        for (int x = q.j; x < Hx; x += a.tpl) {
            T2 c;
            c.x = value(r0, x);
            c.y = value(r1, x);
            lb[x] = c;
            if (x > 0 && x < gx) lb[L - x] = c;
        }
    }
    __syncthreads();
    const T2* out = any_rows<false>(a, m.buf, m.alt, m.twl);
    if (q.line < 0) return;
    for (int k = q.j; k < Hx; k += a.tpl) {
        const T2 v = out[q.line * a.st + k];
        if (r0 < nrows) ghat[int64_t(r0) * Hx + k] = v.x;
        if (r1 < nrows) ghat[int64_t(r1) * Hx + k] = v.y;
    }
}

// Real-even columns as one line (FP64: two), elements p <= L/2 stored.  A last
// column without a partner goes with zeros: whatever stood in the partner's
// place would enter the stored real part, and another block's column may be
// overwritten while it is read.
template <typename T2, typename T> struct AnyEvenColumns {
    T *g0, *g1;
    int ps, L;
    bool on0, on1;
    template <int N> __device__ __forceinline__ void load(int b, int NB, T2 (&v)[N]) const
    {
#pragma unroll
        for (int r = 0; r < N; ++r) {
            const int p = b + r * NB, e = min(p, L - p) * ps;
            v[r].x = g0[e];
            const T y = any_rows_per<T2>() == 2 ? g1[e] : T(0);
            v[r].y = on1 ? y : T(0);
        }
    }
    __device__ __forceinline__ void store1(int p, T2 v) const
    {
        if (2 * p > L) return;
        if (on0) g0[p * ps] = v.x;
        if (on1) g1[p * ps] = v.y;
    }
    template <int N> __device__ __forceinline__ void store(int b, int NB, T2 (&v)[N]) const
    {
#pragma unroll
        for (int r = 0; 2 * r <= N; ++r) store1(b + r * NB, v[r]);
    }
};

template <typename T, int AXIS>
__global__ __launch_bounds__(kAnyThreads, 4) void ga_green_cols(
    const GridJob* __restrict__ jobs, const typename cplx<T>::type* __restrict__ tw, AnyShape a,
    int ncols, int gy, int Hx)
{
    using T2 = typename cplx<T>::type;
    const GridJob& J = jobs[blockIdx.y];
    T* __restrict__ ghat = any_ghat<T>(J);
    const DomainRec* dom = in_memory(J.dom);
    if (dom->error || !dom->ghat_dirty) return;
    AnyLds<T2> m = any_lds(a, tw);
    const AnyLane q = any_lane(a);
    constexpr int W = any_rows_per<T2>();
    const int c0 = W * (any_group() * a.nl + q.line), c1 = W == 2 ? c0 + 1 : ncols;
    const bool on0 = q.line >= 0 && c0 < ncols, on1 = q.line >= 0 && c1 < ncols;
    auto column = [&](int c) {
        const int plane = c / Hx, kx = c - plane * Hx;
        return ghat + int64_t(plane) * (AXIS == 1 ? (gy + 1) * Hx : Hx) + kx;
    };
    const AnyEvenColumns<T2, T> io{column(on0 ? c0 : 0), column(on1 ? c1 : on0 ? c0 : 0),
                                   AXIS == 1 ? Hx : (gy + 1) * Hx, a.pl.L, on0, on1};
    any_columns<false>(a, q, m.buf, m.alt, m.twl, io);
}

// ---------------------------------------------------------------------------
// host: plans, launches
// ---------------------------------------------------------------------------
namespace {

// Threads of a line that take every register pass of a plan in one round.
int line_threads(int L, const std::vector<int>& radices, bool table)
{
    int t = 1;
    for (int r : radices) {
        if (!any_radix(r, table)) continue;
        const int q = any_per(r);
        t = std::max(t, (L / r + q - 1) / q);
    }
    return t;
}

// FP64: fewest radices with product m (at least `least` of them), then the
// fewest threads per line; larger radices first.
void split_length(int L, int m, int most, size_t least, std::vector<int>& cur,
                  std::vector<int>& best)
{
    if (m == 1) {
        if (cur.size() < least) return;
        if (best.empty() || cur.size() < best.size() ||
            line_threads(L, cur, false) < line_threads(L, best, false))
            best = cur;
        return;
    }
    if (!best.empty() && cur.size() >= best.size()) return;
    for (int r = std::min(most, m); r >= 2; --r)
        if (m % r == 0 && any_radix(r, false)) {
            cur.push_back(r);
            split_length(L, m / r, r, least, cur, best);
            cur.pop_back();
        }
}

}  // namespace

AnyPlan any_plan(int L, bool fp32)
{
    AnyPlan p{};
    p.L = L;
    int m = L;
    std::vector<int> radices, rest;
    if (fp32) {
        for (; m % 4 == 0; m /= 4) rest.push_back(4);
        for (int f = 2; m > 1; ++f)
            for (; m % f == 0; m /= f) rest.push_back(f);
        // two passes in one where a composite radix is that pair (a transform
        // keeps a first and a last pass)
        for (size_t k = 0; k < rest.size(); ++k) {
            const int r = k + 1 < rest.size() ? rest[k] * rest[k + 1] : 0;
            const bool pair = r > 0 && r <= 16 && any_split(r) == rest[k] && r / rest[k] == rest[k + 1] &&
                              rest.size() > 2;
            radices.push_back(pair ? r : rest[k]);
            k += pair;
        }
    } else {
        std::vector<int> cur;
        for (int f = 17; f <= m; ++f)  // primes of 17 and more
            for (; m % f == 0 && [f] {
                     for (int d = 2; d * d <= f; ++d)
                         if (f % d == 0) return false;
                     return true;
                 }(); m /= f)
                rest.push_back(f);
        // a transform has a first and a last pass (L is even and at least 8)
        split_length(L, m, 13, rest.empty() ? 2 : 1, cur, radices);
        radices.insert(radices.end(), rest.begin(), rest.end());
    }
    p.tpl = line_threads(L, radices, fp32);
    uint32_t ns = 1;
    for (int r : radices) {
        if (p.np == kAnyMaxPasses) break;  // not reachable for L <= kAnyMaxLen
        p.ns_magic[p.np] = ns > 1 ? div_magic(ns) : 0u;
        p.R[p.np++] = r;
        ns *= uint32_t(r);
    }
    ns = 1;
    for (int k = p.np - 1; k >= 0; --k) {
        p.back_magic[k] = ns > 1 ? div_magic(ns) : 0u;
        ns *= uint32_t(p.R[k]);
    }
    return p;
}

namespace {

inline int64_t nblk(int64_t items, int per) { return (items + per - 1) / per; }

// Blocks of the passes: lines (or pairs) in groups of K transforms.
// Columns: runs of 128 bytes over neighbouring lines; rows: 256 threads.
// Fewer where the threads or the LDS pass their bounds (three blocks on a CU's
// 160 KiB; 40 KiB for four made no difference); one line always fits the 64 KiB
// of a block.
constexpr size_t kAnyLds = 53000;
template <typename T2> AnyShape any_shape(const AnyPlan& pl, int K, bool rows, size_t& lds)
{
    AnyShape a{};
    a.pl = pl;
    int direct = 0;
    for (int s = 0; s < pl.np; ++s) direct |= !any_radix(pl.R[s], any_table<T2>());
    a.two = direct;
    a.st = pl.L | 1;
    auto bytes = [&](int nl) {
        return (size_t(nl) * K * a.st * (a.two ? 2 : 1) + any_periods<T2>() * pl.L) * sizeof(T2);
    };
    // (at most ceil(1022 / 2 / 3) = 171 threads: one line always fits)
    a.tpl = direct ? std::max(pl.tpl, std::min(pl.L / 4, kAnyPreferred / K)) : pl.tpl;
    a.nl = rows ? std::min(16, std::max(1, 256 / (a.tpl * K))) : 128 / int(sizeof(T2));
    while (a.nl > 1 && (a.nl * K * a.tpl > kAnyPreferred || bytes(a.nl) > kAnyLds)) a.nl /= 2;
    a.lines = a.nl * K;
    lds = bytes(a.nl);
    return a;
}

template <typename R> int64_t any_lines(int64_t rows)
{
    return nblk(rows, any_rows_per<typename cplx<R>::type>());
}

template <typename... P, typename... A>
void any_launch(void (*kernel)(P...), bool columns, int64_t lines, int nj, const AnyShape& a,
                size_t lds, hipStream_t st, A... args)
{
    int64_t blocks = nblk(lines, a.nl);
    if (columns) blocks = (blocks + 7) / 8 * 8;
    const int threads = (a.lines * a.tpl + 63) / 64 * 64;
    hipLaunchKernelGGL(kernel, dim3(unsigned(blocks), nj), dim3(threads), lds, st, args...);
}

}  // namespace

template <typename R>
void any_green_x(const Geometry& g, int green_fn, const GridJob* jobs, int nj,
                 const typename cplx<R>::type* tw, hipStream_t st)
{
    size_t lds;
    const AnyShape a = any_shape<typename cplx<R>::type>(g.plan[0], 1, true, lds);
    const int64_t rows = int64_t(g.gz + 1) * (g.gy + 1);
    any_launch(ga_green_x<R>, false, any_lines<R>(rows), nj, a, lds, st, jobs, tw + g.tw_any[0], a,
               g.gx, g.gy, g.gz, green_fn);
}

template <typename R>
void any_green_cols(const Geometry& g, int axis, const GridJob* jobs, int nj,
                    const typename cplx<R>::type* tw, hipStream_t st)
{
    size_t lds;
    const AnyShape a = any_shape<typename cplx<R>::type>(g.plan[axis], 1, false, lds);
    const int cols = (axis == 1 ? (g.gz + 1) : (g.gy + 1)) * g.Hx;
    if (axis == 1)
        any_launch(ga_green_cols<R, 1>, true, any_lines<R>(cols), nj, a, lds, st, jobs,
                   tw + g.tw_any[1], a, cols, g.gy, g.Hx);
    else
        any_launch(ga_green_cols<R, 2>, true, any_lines<R>(cols), nj, a, lds, st, jobs,
                   tw + g.tw_any[2], a, cols, g.gy, g.Hx);
}

template <typename R>
void any_x_pass(const Geometry& g, bool inverse, const GridJob* jobs, int nj,
                const typename cplx<R>::type* tw, hipStream_t st)
{
    using T2 = typename cplx<R>::type;
    size_t lds;
    const AnyShape a = any_shape<T2>(g.plan[0], 1, true, lds);
    const int rows = g.gz * g.gy;
    if (!inverse)
        any_launch(ga_x_r2c<R, false>, false, any_lines<R>(rows), nj, a, lds, st, jobs,
                   tw + g.tw_any[0], a, rows, g.gx, g.gy, g.Dy, static_cast<const R*>(nullptr),
                   static_cast<T2*>(nullptr));
    else
        any_launch(ga_x_c2r<R>, false, any_lines<R>(rows), nj, a, lds, st, jobs, tw + g.tw_any[0], a,
                   rows, g.gx, g.gy, g.Dy);
}

// which: 0 y forward, 1 y inverse, 2 z convolution (the SolveX column passes)
template <typename R>
void any_cols(const Geometry& g, int which, const GridJob* jobs, int nj,
              const typename cplx<R>::type* tw, hipStream_t st)
{
    using T2 = typename cplx<R>::type;
    size_t lds;
    T2* const none = nullptr;
    if (which == 2) {
        const int lines = g.Dy * g.Hx;
        const AnyShape a = any_shape<T2>(g.plan[2], 1, false, lds);
        any_launch(ga_cols<R, 2>, true, lines, nj, a, lds, st, jobs, tw + g.tw_any[2], a, lines,
                   lines, 0, lines, g.gy, g.Hx, none);
        return;
    }
    const int lines = g.gz * g.Hx;
    const AnyShape a = any_shape<T2>(g.plan[1], 1, false, lds);
    const int plane = g.Dy * g.Hx;
    if (which == 0)
        any_launch(ga_cols<R, 0>, true, lines, nj, a, lds, st, jobs, tw + g.tw_any[1], a, lines,
                   g.Hx, plane, g.Hx, g.gy, g.Hx, none);
    else
        any_launch(ga_cols<R, 1>, true, lines, nj, a, lds, st, jobs, tw + g.tw_any[1], a, lines,
                   g.Hx, plane, g.Hx, g.gy, g.Hx, none);
}

// which: 0 z field, 1 y field, 2 x field (the precision form's field passes)
template <typename R>
void any_field(const Geometry& g, int which, const GridJob* jobs, int nj,
               const typename cplx<R>::type* tw, hipStream_t st)
{
    using T2 = typename cplx<R>::type;
    size_t lds;
    if (which == 0) {
        const int lines = g.Dy * g.Hx;
        const AnyShape a = any_shape<T2>(g.plan[2], 2, false, lds);
        any_launch(ga_z_field<R>, true, lines, nj, a, lds, st, jobs, tw + g.tw_any[2], a, lines,
                   g.gy, g.Hx);
    } else if (which == 1) {
        const int lines = g.gz * g.Hx;
        const AnyShape a = any_shape<T2>(g.plan[1], 3, false, lds);
        any_launch(ga_y_field<R>, true, lines, nj, a, lds, st, jobs, tw + g.tw_any[1], a, lines,
                   g.gy, g.Hx);
    } else {
        const AnyShape a = any_shape<T2>(g.plan[0], 3, true, lds);
        any_launch(ga_x_field<R>, false, any_lines<R>(int64_t(g.gz) * g.gy), nj, a, lds, st, jobs, tw + g.tw_any[0], a, g.gx,
                   g.gy, g.gz, g.Dy, div_magic(uint32_t(g.gx)));
    }
}

template <typename R>
void any_chat(const Geometry& g, const void* C, const GridJob* jobs, void* chat_v,
              const typename cplx<R>::type* tw, hipStream_t st)
{
    using T2 = typename cplx<R>::type;
    T2* chat = static_cast<T2*>(chat_v);
    size_t lds;
    // x: every row of the doubled grid, full length Dx
    {
        const AnyShape a = any_shape<T2>(g.plan[0], 1, true, lds);
        const int rows = g.Dz * g.Dy;
        any_launch(ga_x_r2c<R, true>, false, any_lines<R>(rows), 1, a, lds, st, jobs, tw + g.tw_any[0], a,
                   rows, g.gx, g.gy, g.Dy, static_cast<const R*>(C), chat);
    }
    // y: columns of Dy in every plane z < Dz
    {
        const int lines = g.Dz * g.Hx;
        const AnyShape a = any_shape<T2>(g.plan[1], 1, false, lds);
        any_launch(ga_cols<R, 3>, true, lines, 1, a, lds, st, jobs, tw + g.tw_any[1], a, lines,
                   g.Hx, g.Dy * g.Hx, g.Hx, g.gy, g.Hx, chat);
    }
    // z: columns of Dz for every (ky, kx)
    {
        const int lines = g.Dy * g.Hx;
        const AnyShape a = any_shape<T2>(g.plan[2], 1, false, lds);
        any_launch(ga_cols<R, 3>, true, lines, 1, a, lds, st, jobs, tw + g.tw_any[2], a, lines,
                   lines, 0, lines, g.gy, g.Hx, chat);
    }
}

#define SC3D_ANY_INST(R)                                                                       \
    template void any_green_x<R>(const Geometry&, int, const GridJob*, int,                    \
                                 const cplx<R>::type*, hipStream_t);                           \
    template void any_green_cols<R>(const Geometry&, int, const GridJob*, int,                 \
                                    const cplx<R>::type*, hipStream_t);                        \
    template void any_x_pass<R>(const Geometry&, bool, const GridJob*, int,                    \
                                const cplx<R>::type*, hipStream_t);                            \
    template void any_cols<R>(const Geometry&, int, const GridJob*, int, const cplx<R>::type*, \
                              hipStream_t);                                                    \
    template void any_chat<R>(const Geometry&, const void*, const GridJob*, void*,            \
                              const cplx<R>::type*, hipStream_t);
SC3D_ANY_INST(double)
SC3D_ANY_INST(float)
template void any_field<float>(const Geometry&, int, const GridJob*, int, const float2*,
                               hipStream_t);
#undef SC3D_ANY_INST

}  // namespace sc3d
