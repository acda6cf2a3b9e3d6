// sc3d_particles.hip -- particle-side kernels of the MI355X space-charge step:
// bunch extent, cell keys + stable radix sort + in-place reorder, CIC
// deposit, E field, gather-interpolate-kick, and the Gaussian populate.
#include "sc3d_particles.h"

namespace sc3d {

// ---------------------------------------------------------------------------
// Served form: opens one apply of a scheduled job (see StepCtl).  Schedule
// table layout: [first | between | last], turn_steps programs each; step j
// of the job is schedule entry k = j mod turn_steps; the maps before the
// kick run on the first step only, and the program fused after the kick is
// between[k] (the second half-step of k and the first of k+1) except after
// the last step (last[k]).
// ---------------------------------------------------------------------------
__global__ void k_step_begin(StepCtl* __restrict__ ctl)
{
    if (threadIdx.x != 0 || blockIdx.x != 0) return;
    StepCtl c = *ctl;
    const int64_t j = c.applies;
    if (c.turn_steps > 0 && j >= c.total_steps) {
        c.done = 1;
        *ctl = c;
        return;
    }
    c.done = 0;
    if (c.turn_steps > 0) {
        const int k = int(j % c.turn_steps);
        c.cur = k;
        c.first_prog = j == 0 ? k : -1;
        c.after_prog = j < c.total_steps - 1 ? c.turn_steps + k : 2 * c.turn_steps + k;
    }
    c.applies = j + 1;
    *ctl = c;
}

// ---------------------------------------------------------------------------
// Bunch extent: the six sums of Core_diagnostics::calculate_spatial_mean_stddev
// (core_diagnostics.cc:139-153) in one fixed tree, identical for every launch
// configuration and device:
//   chunk c = particles [4096c, 4096c+4096); lane t adds, from +0.0 and in
//   order j = 0..15, particle 4096c + 256j + t (masked and >= n skipped);
//   lanes combine pairwise (s[t] += s[t+w], w = 1..128), first inside each
//   64-wide wavefront by xor butterflies, then across the four wavefronts;
//   chunk partials combine by the same rule in k_domain_finish.
// ---------------------------------------------------------------------------
__device__ __forceinline__ double wave_pairwise_sum(double v);

__device__ __forceinline__ void block_pairwise6(double (&s)[6], double (*ws)[6])
{
#pragma unroll
    for (int q = 0; q < 6; ++q) s[q] = wave_pairwise_sum(s[q]);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0)
#pragma unroll
        for (int q = 0; q < 6; ++q) ws[wave][q] = s[q];
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int q = 0; q < 6; ++q) s[q] = (ws[0][q] + ws[1][q]) + (ws[2][q] + ws[3][q]);
}

template <int K>
__device__ __forceinline__ void block_pairwiseK(double (&s)[K], double (*ws)[K])
{
#pragma unroll
    for (int q = 0; q < K; ++q) s[q] = wave_pairwise_sum(s[q]);
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    if (lane == 0)
#pragma unroll
        for (int q = 0; q < K; ++q) ws[wave][q] = s[q];
    __syncthreads();
    if (threadIdx.x == 0)
#pragma unroll
        for (int q = 0; q < K; ++q) s[q] = (ws[0][q] + ws[1][q]) + (ws[2][q] + ws[3][q]);
}

// Moments for diagnostics (Core_diagnostics::calculate_mean / calculate_mom2,
// core_diagnostics.cc:126-198,202-229,318-362): MODE 0 sums the six
// coordinates; MODE 1 sums the 21 centred products (p_j - mean_j)(p_k -
// mean_k), k <= j, with the mean read from `mean`.  Same fixed tree as the
// bunch extent (chunks of 4096, 16 per lane, pairwise lanes).
template <int MODE>
__global__ __launch_bounds__(kThreads) void k_moments_partial(const double* __restrict__ parts,
                                                              int64_t stride,
                                                              const uint8_t* __restrict__ masks,
                                                              int64_t n,
                                                              const double* __restrict__ mean,
                                                              double* __restrict__ P)
{
    constexpr int K = MODE == 0 ? 6 : 21;
    __shared__ double ws[4][K];
    double s[K];
#pragma unroll
    for (int q = 0; q < K; ++q) s[q] = 0.0;
    double m[6] = {0, 0, 0, 0, 0, 0};
    if (MODE == 1)
        for (int j = 0; j < 6; ++j) m[j] = mean[j];
    // four rounds' loads are issued before their sums (none waits for a mask)
    constexpr int U = 4;
    const int64_t c = blockIdx.x;
    for (int j0 = 0; j0 < 16; j0 += U) {
        double v[U][6];
        uint8_t on[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = c * 4096 + int64_t(j0 + u) * 256 + threadIdx.x;
            on[u] = 0;
            if (i < n) {
                on[u] = masks[i];
#pragma unroll
                for (int j = 0; j < 6; ++j) v[u][j] = parts[i + j * stride];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u) {
            if (!on[u]) continue;
            if (MODE == 0) {
#pragma unroll
                for (int j = 0; j < 6; ++j) s[j] += v[u][j];
            } else {
                int q = 0;
#pragma unroll
                for (int j = 0; j < 6; ++j) {
                    const double dj = v[u][j] - m[j];
#pragma unroll
                    for (int k = 0; k <= j; ++k) s[q++] += dj * (v[u][k] - m[k]);
                }
            }
        }
    }
    block_pairwiseK<K>(s, ws);
    if (threadIdx.x == 0)
        for (int q = 0; q < K; ++q) P[c * K + q] = s[q];
}

// Combines the chunk partials by the same rule and divides by total_num, one
// sum per block: each lane's chain is then one load per 256 chunks (4 at 4e6
// particles), where one block for all K sums took 4.6 / 9.0 us (K = 6 / 21).
template <int K>
__global__ __launch_bounds__(kThreads) void k_moments_finish(const double* __restrict__ P,
                                                             int64_t nch, double total_num,
                                                             double* __restrict__ out)
{
    __shared__ double ws[4][1];
    const int q = blockIdx.x;
    double s[1] = {0.0};
    for (int64_t c = threadIdx.x; c < nch; c += kThreads) s[0] += P[c * K + q];
    block_pairwiseK<1>(s, ws);
    if (threadIdx.x == 0) out[q] = s[0] / total_num;
}

// ---------------------------------------------------------------------------
// Tail counts (diagnostic of the halo comparison of long tracking): per
// plane j, active particles with |p_j - c_j| > lim_j.  Integer counts, so
// the result does not depend on the reduction order.  Every block stores its
// counts and a second launch sums them: per-wavefront atomics (6 x 8192 on
// one cache line, about 12 ns each) held the pass at 610 us at 4e6 particles;
// now 32 us, 49 bytes per particle at 6.2 TB/s.
// (A block counts n / 1024 particles: 32 bits hold it.)
// ---------------------------------------------------------------------------
__global__ __launch_bounds__(kThreads) void k_tail_counts(const double* __restrict__ parts,
                                                          int64_t stride,
                                                          const uint8_t* __restrict__ masks,
                                                          int64_t n, TailArgs a,
                                                          uint32_t* __restrict__ partial)
{
    __shared__ uint32_t ws[kThreads / 64][6];
    uint32_t cnt[6] = {0u, 0u, 0u, 0u, 0u, 0u};
    constexpr int U = 4;  // rounds in flight
    const int64_t T = int64_t(gridDim.x) * kThreads;
    for (int64_t i0 = blockIdx.x * int64_t(kThreads) + threadIdx.x; i0 < n; i0 += U * T) {
        double v[U][6];
        uint8_t on[U];
#pragma unroll
        for (int u = 0; u < U; ++u) {
            const int64_t i = i0 + u * T;
            on[u] = 0;
            if (i < n) {
                on[u] = masks[i];
#pragma unroll
                for (int j = 0; j < 6; ++j) v[u][j] = parts[i + j * stride];
            }
        }
#pragma unroll
        for (int u = 0; u < U; ++u)
            if (on[u])
#pragma unroll
                for (int j = 0; j < 6; ++j) cnt[j] += fabs(v[u][j] - a.c[j]) > a.lim[j];
    }
#pragma unroll
    for (int j = 0; j < 6; ++j) {
#pragma unroll
        for (int w = 1; w < 64; w *= 2) cnt[j] += __shfl_xor(cnt[j], w, 64);
        if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6][j] = cnt[j];
    }
    __syncthreads();
    if (threadIdx.x < 6) {
        uint32_t t = 0;
        for (int w = 0; w < kThreads / 64; ++w) t += ws[w][threadIdx.x];
        partial[threadIdx.x * kTailBlocks + blockIdx.x] = t;
    }
}

// Sums the blocks' counts, one plane per block.
__global__ __launch_bounds__(kThreads) void k_tail_finish(const uint32_t* __restrict__ partial,
                                                          int nblk,
                                                          unsigned long long* __restrict__ counts)
{
    __shared__ unsigned long long ws[kThreads / 64];
    unsigned long long t = 0;
    for (int b = threadIdx.x; b < nblk; b += kThreads)
        t += partial[blockIdx.x * kTailBlocks + b];
#pragma unroll
    for (int w = 1; w < 64; w *= 2) t += __shfl_xor(t, w, 64);
    if ((threadIdx.x & 63) == 0) ws[threadIdx.x >> 6] = t;
    __syncthreads();
    if (threadIdx.x == 0) {
        for (int w = 1; w < kThreads / 64; ++w) t += ws[w];
        counts[blockIdx.x] = t;
    }
}

void launch_moments(const double* parts, int64_t stride, const uint8_t* masks, int64_t n,
                    double total_num, double* P, double* out /* 6 + 21 */, hipStream_t st)
{
    int64_t nch = (n + 4095) / 4096;
    if (nch > 0)
        hipLaunchKernelGGL(k_moments_partial<0>, dim3(unsigned(nch)), dim3(kThreads), 0, st,
                           parts, stride, masks, n, (const double*)nullptr, P);
    hipLaunchKernelGGL(k_moments_finish<6>, dim3(6), dim3(kThreads), 0, st, P, nch, total_num,
                       out);
    if (nch > 0)
        hipLaunchKernelGGL(k_moments_partial<1>, dim3(unsigned(nch)), dim3(kThreads), 0, st,
                           parts, stride, masks, n, (const double*)out, P);
    hipLaunchKernelGGL(k_moments_finish<21>, dim3(21), dim3(kThreads), 0, st, P, nch, total_num,
                       out + 6);
}

// space_charge_3d_open_hockney.cc:94-109
__device__ double smallest_non_tiny(double val, double o1, double o2, double tiny)
{
    if (val > tiny) return val;
    if ((o1 > tiny) && (o2 > tiny)) return fmin(o1, o2);
    return fmax(o1, o2);
}

// Finishes the domain on the device (update_domain, .cc:493-540, with the
// host finish of core_diagnostics.cc:454-459 and Rectangular_grid_domain,
// rectangular_grid_domain.h:20-36) and derives weight0 (deposit.cc:608-610),
// the force normalisation (.cc:707-735) and the kick factor (.cc:759-770).
// Also decides whether the cached Green's spectrum is still valid (same h
// bits) or must be recomputed this step.
__global__ __launch_bounds__(kThreads) void k_domain_finish(const double* __restrict__ P,
                                                            int64_t nch, DomainFinishArgs a,
                                                            DomainRec* __restrict__ dom, Sched sc)
{
    __shared__ double ws[4][6];
    if (sc.ctl) {
        // served form: a finished job's applies do nothing; the kick time
        // step comes from the schedule
        if (sc.ctl->done) {
            if (threadIdx.x == 0) dom->error = kDoneMark;
            return;
        }
        if (sc.ctl->turn_steps > 0) a.time_step = sc.dt[sc.ctl->cur];
    }
    double s[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    if (!a.fixed) {
        // lane t adds chunks t, t + 256, ... in order; eight chunks' loads are
        // issued before their adds
        constexpr int U = 8;
        for (int64_t c0 = threadIdx.x; c0 < nch; c0 += U * kThreads) {
            double v[U][6];
#pragma unroll
            for (int u = 0; u < U; ++u) {
                const int64_t c = c0 + int64_t(u) * kThreads;
                if (c < nch)
#pragma unroll
                    for (int q = 0; q < 6; ++q) v[u][q] = P[c * 6 + q];
            }
#pragma unroll
            for (int u = 0; u < U; ++u)
                if (c0 + int64_t(u) * kThreads < nch)
#pragma unroll
                    for (int q = 0; q < 6; ++q) s[q] += v[u][q];
        }
        block_pairwise6(s, ws);
    }
    if (threadIdx.x != 0) return;
    DomainRec d = *dom;  // keeps the Green's cache fields
    double size[3], offset[3];
    d.error = 0;
    d.rho_peak = 0;
    if (a.fixed) {
        for (int k = 0; k < 3; ++k) {
            size[k] = a.size[k];
            offset[k] = a.offset[k];
            d.sums[k] = d.sums[k + 3] = 0.0;
            d.mean[k] = d.stddev[k] = 0.0;
        }
    } else {
        for (int q = 0; q < 6; ++q) d.sums[q] = s[q];
        for (int j = 0; j < 3; ++j) {
            d.mean[j] = s[j] / a.total_num;
            d.stddev[j] = sqrt(s[j + 3] / a.total_num - d.mean[j] * d.mean[j]);
        }
        const double tiny = 1.0e-10;
        if ((d.stddev[0] < tiny) && (d.stddev[1] < tiny) && (d.stddev[2] < tiny)) {
            d.error = SC3D_ERR_DOMAIN;
            d.ghat_dirty = 0;
            *dom = d;
            return;
        }
        offset[0] = d.mean[0];
        offset[1] = d.mean[1];
        offset[2] = d.mean[2];
        size[0] = a.n_sigma * smallest_non_tiny(d.stddev[0], d.stddev[1], d.stddev[2], tiny);
        size[1] = a.n_sigma * smallest_non_tiny(d.stddev[1], d.stddev[0], d.stddev[2], tiny);
        size[2] = a.n_sigma * smallest_non_tiny(d.stddev[2], d.stddev[0], d.stddev[1], tiny);
        if (a.grid_entire_period) {
            offset[2] = 0.0;
            size[2] = a.z_period;
        }
    }
    for (int k = 0; k < 3; ++k) {
        d.size[k] = size[k];
        d.offset[k] = offset[k];
        d.left[k] = offset[k] - size[k] / 2.0;
        d.h[k] = size[k] / (1.0 * a.shape[k]);
        d.inv_h[k] = 1.0 / d.h[k];
        d.half_inv_h[k] = 0.5 / d.h[k];
    }
    const double* h = d.h;
    d.w0 = (a.real_num / a.total_num) * a.charge * kE / (h[0] * h[1] * h[2]);
    double norm = h[0] * h[1] * h[2];
    norm *= 1.0 / (4.0 * kPi * kEpsilon0);
    norm *= 1.0;
    if (a.green_fn == SC3D_GREEN_LINEAR) norm *= 1.0 / (h[2] * h[2]);
    norm *= 1.0 / (2 * a.shape[0] * 2 * a.shape[1] * 2 * a.shape[2]);
    d.fn_norm = norm;
    double q = a.charge * kE;
    double unit_conversion = kC / (1e9 * kE);
    d.factor = a.kick_scale * unit_conversion * q * a.time_step * d.fn_norm /
               (a.ref_p * a.ref_gamma * a.ref_gamma * a.ref_beta);
    bool same = d.ghat_valid && __double_as_longlong(d.ghat_h[0]) == __double_as_longlong(h[0]) &&
                __double_as_longlong(d.ghat_h[1]) == __double_as_longlong(h[1]) &&
                __double_as_longlong(d.ghat_h[2]) == __double_as_longlong(h[2]);
    d.ghat_dirty = same ? 0 : 1;
    for (int k = 0; k < 3; ++k) d.ghat_h[k] = h[k];
    d.ghat_valid = 1;
    *dom = d;
}

// The chunk sums and the clearing of the density grid in one launch: every
// block clears its slice of the grid (16-byte stores; the grid of the
// previous apply was consumed by its solve) and writes its chunk partials.
// (Finishing in the last block to count itself in, behind device-scope
// fences, measured slower: 41 against 25 us per apply at 4e6 particles, the
// fence of each of the 977 blocks writing back its L2.)
__global__ __launch_bounds__(kThreads) void k_domain_partial(
    const double* __restrict__ parts, int64_t stride, const uint8_t* __restrict__ masks,
    int64_t n, double* __restrict__ P, const StepCtl* __restrict__ ctl, uint4* __restrict__ grid,
    int64_t grid16)
{
    __shared__ double ws[4][6];
    if (ctl && ctl->done) return;
    if (grid16 > 0) {
        const int64_t per = (grid16 + gridDim.x - 1) / gridDim.x;
        const int64_t g0 = int64_t(blockIdx.x) * per;
        const int64_t g1 = g0 + per < grid16 ? g0 + per : grid16;
        for (int64_t i = g0 + threadIdx.x; i < g1; i += kThreads) grid[i] = make_uint4(0, 0, 0, 0);
    }
    double s[6] = {0.0, 0.0, 0.0, 0.0, 0.0, 0.0};
    const int64_t i0 = int64_t(blockIdx.x) * 4096 + threadIdx.x;
    // Four rounds' loads ahead of the four summed, no branch between them (a
    // lane past n reads the last particle): an inactive particle adds +0.0,
    // which changes no sum (none is ever -0.0).
    constexpr int kAhead = 4;
    double x[2][kAhead], y[2][kAhead], z[2][kAhead];
    uint8_t on[2][kAhead];
    auto load = [&](int b) {
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            const int64_t i = min(i0 + int64_t(b * kAhead + j) * 256, n - 1);
            on[b & 1][j] = masks[i];
            x[b & 1][j] = parts[i];
            y[b & 1][j] = parts[i + 2 * stride];
            z[b & 1][j] = parts[i + 4 * stride];
        }
    };
    load(0);
#pragma unroll
    for (int b = 0; b < 16 / kAhead; ++b) {
        if (b + 1 < 16 / kAhead) load(b + 1);
#pragma unroll
        for (int j = 0; j < kAhead; ++j) {
            const bool in = on[b & 1][j] != 0 && i0 + int64_t(b * kAhead + j) * 256 < n;
            const double px = in ? x[b & 1][j] : 0.0;
            const double py = in ? y[b & 1][j] : 0.0;
            const double pz = in ? z[b & 1][j] : 0.0;
            s[0] += px;
            s[1] += py;
            s[2] += pz;
            s[3] += px * px;
            s[4] += py * py;
            s[5] += pz * pz;
        }
    }
    block_pairwise6(s, ws);
    if (threadIdx.x == 0)
        for (int q = 0; q < 6; ++q) P[int64_t(blockIdx.x) * 6 + q] = s[q];
}

// ---------------------------------------------------------------------------
// Cell keys in brick order: the cells are grouped in bricks of 4 cells per
// axis (an axis whose length 4 does not divide keeps bricks of 1 there).
// The bricks follow a serpentine path, x fastest: rows of bricks run
// backwards in x on odd rows (counting rows r = bz*nby + by'), and the rows
// of a layer run backwards in y on odd layers bz (by' = nby-1-by), so
// consecutive bricks are always face neighbours; the cells of one brick are
// in (z, y, x) order:
//   k = (r*nbx + bx') * |brick| + (lz*By + ly)*Bx + lx,
// a bijection of the cells onto [0, G).  Active particles with lower corner
// in [0, g-2]^3 (the particles the deposit and the kick touch) get their
// cell's key, the rest G.  A window of consecutive particles of this order
// spans a compact box of cells: the deposit's and the kick's node tiles, and
// the reorder's reads, stay local.
// ---------------------------------------------------------------------------
constexpr int kBrickLog2 = 2;  // 4 cells per axis

// log2 of the brick length along an axis of g cells
__device__ __forceinline__ int brick_log2(int g)
{
    return (g & ((1 << kBrickLog2) - 1)) == 0 ? kBrickLog2 : 0;
}

__device__ __forceinline__ int32_t brick_key(int ix, int iy, int iz, int gx, int gy, int gz)
{
    const int sx = brick_log2(gx), sy = brick_log2(gy), sz = brick_log2(gz);
    const int nbx = gx >> sx, nby = gy >> sy, bz = iz >> sz;
    int by = iy >> sy, bx = ix >> sx;
    if (bz & 1) by = nby - 1 - by;  // layers of odd bz: rows backwards
    const int row = bz * nby + by;
    if (row & 1) bx = nbx - 1 - bx;  // odd rows: bricks backwards
    const int brick = row * nbx + bx;
    const int cell = (((iz & ((1 << sz) - 1)) << sy) + (iy & ((1 << sy) - 1))) << sx |
                     (ix & ((1 << sx) - 1));
    return (brick << (sx + sy + sz)) + cell;
}

__device__ __forceinline__ int32_t cell_key(bool active, double x, double y, double z, int gx,
                                            int gy, int gz, const DomainRec& d)
{
    double o;
    int ix, iy, iz;
    const bool in_x = grid_cell(x, d.left[0], d.inv_h[0], gx, ix, o);
    const bool in_y = grid_cell(y, d.left[1], d.inv_h[1], gy, iy, o);
    const bool in_z = grid_cell(z, d.left[2], d.inv_h[2], gz, iz, o);
    const int32_t key = brick_key(ix, iy, iz, gx, gy, gz);
    return (active & in_x & in_y & in_z) ? key : gx * gy * gz;
}

// ---------------------------------------------------------------------------
// Stable LSD radix sort of (key, index): tiles of 256 lanes x ITEMS rounds,
// digits of up to 8 bits, or of 9 where that takes fewer passes.  In
// the scatter, equal digits inside a wavefront are matched with `width`
// ballots, so ranks need one LDS update per distinct digit per wavefront.
// ---------------------------------------------------------------------------
constexpr int kMaxDigitBits = 8;
constexpr int kWideDigitBits = 9;

// lanes of this wavefront holding the same digit (valid lanes only)
__device__ __forceinline__ uint64_t match_digit(int d, bool valid, int width)
{
    const uint64_t v = __ballot(valid);
    uint32_t lo = uint32_t(v), hi = uint32_t(v >> 32);
#pragma unroll 2
    for (int b = 0; b < width; ++b) {
        const int32_t bit = __builtin_amdgcn_sbfe(d, b, 1);  // 0 or -1
        const uint64_t m = __ballot(bit);
        lo &= ~(uint32_t(m) ^ uint32_t(bit));
        hi &= ~(uint32_t(m >> 32) ^ uint32_t(bit));
    }
    return uint64_t(hi) << 32 | lo;
}

#ifndef SC3D_XCD_PART
#define SC3D_XCD_PART 1
#endif

// Block index of this workgroup in an XCD-contiguous order.  Workgroups of
// a launch go to the 8 XCDs round-robin (workgroup b to XCD b % 8) and each
// XCD has its own L2; renumbered so that XCD x runs the x-th eighth of the
// blocks, neighbouring tiles (whose partial cache lines of the sort output,
// the digit counts and the reorder buffers meet) share one L2.  Used by the
// sort and reorder kernels (measured faster); the deposit and the kick keep
// the dispatch order (measured slower with it).  Grids are rounded up to
// multiples of 8 by the launchers; any other grid keeps the identity.
__device__ __forceinline__ unsigned part_block()
{
#if SC3D_XCD_PART
    const unsigned nb = gridDim.x, b = blockIdx.x;
    if ((nb & 7u) == 0u) return (b & 7u) * (nb >> 3) + (b >> 3);
#endif
    return blockIdx.x;
}

// A particle for the deposit through a permutation, which reads in random
// order: one 32-byte read instead of one line in each of three columns and the
// masks.  Written by the key pass.
struct alignas(32) Packed {
    double x, y, z, active;
};

// The per-tile digit counts: entry (digit d, tile b), digit-major (the scan
// reads a digit's row contiguously; measured faster than tile-major rows,
// whose column reads in the scan cost more than the count pass's scattered
// stores save: sort phase 175 vs 183 us at 4e6 particles, 654 vs 683 us at
// 1.6e7).
__device__ __forceinline__ int64_t count_at(int d, int64_t b, int nblk)
{
    return int64_t(d) * nblk + b;
}

// Lane moves inside the register file (DPP, GFX9 controls) for the
// wavefront scans, instead of LDS permutes: rows of 16 lanes; a lane with no
// source lane, or in a row outside ROW_MASK, returns `old`.
constexpr int kDppRowShr = 0x110;  // + n: from lane - n of the same row
constexpr int kDppRowBcast15 = 0x142;  // lane 15 of each row to the next row
constexpr int kDppRowBcast31 = 0x143;  // lane 31 to rows 2 and 3
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ int dpp_move(int old, int v)
{
    return __builtin_amdgcn_update_dpp(old, v, CTRL, ROW_MASK, 0xf, false);
}
template <int CTRL, int ROW_MASK = 0xf>
__device__ __forceinline__ double dpp_move(double old, double v)
{
    const long long o = __double_as_longlong(old), x = __double_as_longlong(v);
    const unsigned lo = unsigned(dpp_move<CTRL, ROW_MASK>(int(o), int(x)));
    const int hi = dpp_move<CTRL, ROW_MASK>(int(o >> 32), int(x >> 32));
    return __longlong_as_double((long long)(uint64_t(lo) | (uint64_t(unsigned(hi)) << 32)));
}

// The xor-butterfly sum of one double per lane (s[t] += s[t ^ w], w = 1, 2,
// .., 32) as lane 0 forms it, in every lane.  After the step of w every
// lane of a group of 2w holds the same value, so any lane of the partner
// group serves: w = 1, 2 by quad permutes, 4 by the half-row mirror, 8 by
// the row mirror (DPP moves), and the rows' totals a, b, c, d (lanes 0, 16,
// 32, 48) combine as lane 0 combines them, (a + b) + (c + d).  Every lane of
// the wavefront calls it.  (Against six ds_bpermute exchanges per value:
// domain phase 25.0 -> 24.5 us at 4e6, 103.3 -> 102.2 us at 1.6e7.)
constexpr int kDppQuadXor1 = 0xB1;       // quad_perm [1, 0, 3, 2]
constexpr int kDppQuadXor2 = 0x4E;       // quad_perm [2, 3, 0, 1]
constexpr int kDppRowMirror = 0x140;
constexpr int kDppRowHalfMirror = 0x141;
__device__ __forceinline__ double readlane_f64(double v, int lane)
{
    const long long x = __double_as_longlong(v);
    const unsigned lo = unsigned(__builtin_amdgcn_readlane(int(x), lane));
    const unsigned hi = unsigned(__builtin_amdgcn_readlane(int(x >> 32), lane));
    return __longlong_as_double((long long)(uint64_t(lo) | (uint64_t(hi) << 32)));
}
__device__ __forceinline__ double wave_pairwise_sum(double v)
{
    v = v + dpp_move<kDppQuadXor1>(v, v);
    v = v + dpp_move<kDppQuadXor2>(v, v);
    v = v + dpp_move<kDppRowHalfMirror>(v, v);
    v = v + dpp_move<kDppRowMirror>(v, v);
    return (readlane_f64(v, 0) + readlane_f64(v, 16)) + (readlane_f64(v, 32) + readlane_f64(v, 48));
}

// Exclusive prefix of one value per thread over the block (DPP lane moves
// inside each wavefront, one LDS exchange of the wavefront sums); every
// thread of the block calls it.  `wsum` holds kThreads/64 entries; callers
// separate two uses by a barrier.
__device__ __forceinline__ int32_t block_exclusive_scan(int32_t v, int32_t* wsum, int32_t& total)
{
    constexpr int kWaves = kThreads / 64;
    const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
    // inclusive wavefront scan: inside rows of 16 lanes, then across rows
    int32_t x = v;
    x += dpp_move<kDppRowShr + 1>(0, x);
    x += dpp_move<kDppRowShr + 2>(0, x);
    x += dpp_move<kDppRowShr + 4>(0, x);
    x += dpp_move<kDppRowShr + 8>(0, x);
    x += dpp_move<kDppRowBcast15, 0xa>(0, x);
    x += dpp_move<kDppRowBcast31, 0xc>(0, x);
    if (lane == 63) wsum[wave] = x;
    __syncthreads();
    int32_t off = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < kWaves; ++w) {
        const int32_t ws = wsum[w];
        off += w < wave ? ws : 0;
        tot += ws;
    }
    total = tot;
    return off + x - v;
}

// Histogram of one digit per tile.  Every lane first loads (or, with KEYS,
// computes from the particles and stores) its keys, so all loads of the
// tile are in flight together; each wavefront then counts its quarter of
// the tile into its own LDS histogram, one update per distinct digit and
// round (ballot match: after the first pass equal digits cluster), and the
// four are summed.  KEYS fuses the key pass into pass 0.  WIDTH: largest
// digit width taken.
template <bool KEYS, int ITEMS, int WIDTH>
__global__ __launch_bounds__(kThreads) void k_radix_count(
    const double* __restrict__ parts, int64_t stride, const uint8_t* __restrict__ masks, int gx,
    int gy, int gz, int32_t* __restrict__ keys, int64_t n, int shift, int width,
    int32_t* __restrict__ counts, int nblk, const DomainRec* __restrict__ dom,
    Packed* __restrict__ packed)
{
    constexpr int kWaves = kThreads / 64;
    constexpr int kTile = kThreads * ITEMS;
    constexpr int kWaveItems = kTile / kWaves;
    constexpr int kPer = (1 << WIDTH) / kThreads;  // digits per thread
    __shared__ int32_t hist[kWaves][1 << WIDTH];
    if (dom->error) return;
    const unsigned blk = part_block();
    if (blk >= unsigned(nblk)) return;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int nb = 1 << width;
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
#pragma unroll
        for (int q = 0; q < kPer; ++q) hist[w][q * kThreads + t] = 0;
    const int64_t base = int64_t(blk) * kTile + int64_t(wave) * kWaveItems;
    int32_t kk[ITEMS];
    if (KEYS) {
        const DomainRec d = *dom;
        constexpr int kBatch = 4;  // particles loaded ahead (a lane past n reads the last one)
#pragma unroll
        for (int r0 = 0; r0 < ITEMS; r0 += kBatch) {
            double x[kBatch], y[kBatch], z[kBatch];
            uint8_t m[kBatch];
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const int64_t i = min(base + (r0 + j) * 64 + lane, n - 1);
                x[j] = parts[i];
                y[j] = parts[i + 2 * stride];
                z[j] = parts[i + 4 * stride];
                m[j] = masks[i];
            }
#pragma unroll
            for (int j = 0; j < kBatch; ++j) {
                const int64_t i = base + (r0 + j) * 64 + lane;
                const int32_t key = cell_key(m[j] != 0, x[j], y[j], z[j], gx, gy, gz, d);
                kk[r0 + j] = i < n ? key : -1;
                if (i < n) {
                    keys[i] = key;
                    if (packed) packed[i] = Packed{x[j], y[j], z[j], m[j] ? 1.0 : 0.0};
                }
            }
        }
    } else {
#pragma unroll
        for (int r = 0; r < ITEMS; ++r) {
            const int64_t i = base + r * 64 + lane;
            kk[r] = i < n ? keys[i] : -1;  // keys are >= 0
        }
    }
    __syncthreads();
    const uint64_t lt_mask = (1ull << lane) - 1;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const bool valid = kk[r] >= 0;
        const int dg = (kk[r] >> shift) & (nb - 1);
        const uint64_t peers = match_digit(dg, valid, width);
        if (valid && __popcll(peers & lt_mask) == 0) hist[wave][dg] += __popcll(peers);
    }
    __syncthreads();
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const int d = q * kThreads + t;
        if (d >= nb) break;
        int32_t c = 0;
#pragma unroll
        for (int w = 0; w < kWaves; ++w) c += hist[w][d];
        counts[count_at(d, blk, nblk)] = c;
    }
}

// One block per digit: exclusive scan of that digit's per-tile counts (in
// place) and the digit total.
__global__ __launch_bounds__(kThreads) void k_radix_scan(int32_t* __restrict__ counts, int nblk,
                                                         int32_t* __restrict__ totals,
                                                         const DomainRec* dom)
{
    __shared__ int32_t wsum[kThreads / 64];
    if (dom->error) return;
    const int d = blockIdx.x;
    const int per = (nblk + kThreads - 1) / kThreads;
    const int b0 = threadIdx.x * per;
    int32_t s = 0;
    for (int k = 0; k < per; ++k)
        if (b0 + k < nblk) s += counts[count_at(d, b0 + k, nblk)];
    int32_t total;
    int32_t run = block_exclusive_scan(s, wsum, total);
    for (int k = 0; k < per; ++k)
        if (b0 + k < nblk) {
            const int64_t at = count_at(d, b0 + k, nblk);
            const int32_t v = counts[at];
            counts[at] = run;
            run += v;
        }
    if (threadIdx.x == 0) totals[d] = total;
}

// Stable scatter of one tile.  Wavefront w ranks the w-th quarter of the
// tile's items in ITEMS rounds of 64 with wave-private
// digit counters (ballot match: rank among equal digits of the round, the
// lowest lane of each digit group advances the counter), with no block
// barrier inside the rounds.  The tile's digit counts come from the count
// pass (difference of consecutive exclusive prefixes).  Every item is then
// placed in LDS at its position in the tile's stable digit order, and the
// tile is written out in that order, so each digit's items of the tile form
// one contiguous run in the output (positions as a per-item scatter would
// give them).
template <int ITEMS, int WIDTH>
__global__ __launch_bounds__(kThreads) void k_radix_scatter(
    const int32_t* __restrict__ keys_in, const int32_t* __restrict__ vals_in, int64_t n,
    int shift, int width, const int32_t* __restrict__ counts, const int32_t* __restrict__ totals,
    int nblk, int32_t* __restrict__ keys_out, int32_t* __restrict__ vals_out,
    const DomainRec* dom)
{
    constexpr int kWaves = kThreads / 64;
    constexpr int kTile = kThreads * ITEMS;
    constexpr int kWaveItems = kTile / kWaves;
    constexpr int kPer = (1 << WIDTH) / kThreads;  // digits per thread, consecutive
    __shared__ int32_t delta[1 << WIDTH];  // output position of a digit's items less that in the tile
    __shared__ int32_t wave_off[kWaves][1 << WIDTH];
    __shared__ int32_t wsum[2][kWaves];
    __shared__ int32_t lkey[kTile];
    __shared__ int32_t lval[kTile];
    if (dom->error) return;
    const unsigned blk = part_block();
    if (blk >= unsigned(nblk)) return;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int nb = 1 << width;
    const int64_t tile = int64_t(blk) * kTile;
    const int nvalid = int(n - tile < kTile ? n - tile : kTile);
    // all of the tile's loads in flight together
    int32_t kk[ITEMS], vv[ITEMS], rk[ITEMS];
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const int64_t i = tile + int64_t(wave) * kWaveItems + r * 64 + lane;
        kk[r] = i < n ? keys_in[i] : -1;  // keys are >= 0; -1 marks lanes past n
        vv[r] = i < n ? (vals_in ? vals_in[i] : int32_t(i)) : 0;
    }
    // digit totals -> exclusive prefix over digits (global digit bases);
    // this tile's digit counts -> local digit starts
    int32_t tot[kPer], cnt[kPer], before[kPer], tsum = 0, csum = 0;
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        const int d = t * kPer + q;
        tot[q] = cnt[q] = before[q] = 0;
        if (d < nb) {
            tot[q] = totals[d];
            before[q] = counts[count_at(d, blk, nblk)];
            cnt[q] = (blk + 1 < unsigned(nblk) ? counts[count_at(d, blk + 1, nblk)] : tot[q]) -
                     before[q];
        }
        tsum += tot[q];
        csum += cnt[q];
    }
    int32_t all_n, tile_n;
    int32_t digit_base = block_exclusive_scan(tsum, wsum[0], all_n);
    int32_t local_start = block_exclusive_scan(csum, wsum[1], tile_n);
    int32_t start[kPer];
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        start[q] = local_start;
        delta[t * kPer + q] = digit_base + before[q] - local_start;
        digit_base += tot[q];
        local_start += cnt[q];
    }
#pragma unroll
    for (int w = 0; w < kWaves; ++w)
#pragma unroll
        for (int q = 0; q < kPer; ++q) wave_off[w][q * kThreads + t] = 0;
    __syncthreads();
    // ranking inside each wavefront's quarter of the tile
    const uint64_t lt_mask = (1ull << lane) - 1;
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        const bool valid = kk[r] >= 0;
        const int dg = (kk[r] >> shift) & (nb - 1);
        const uint64_t peers = match_digit(dg, valid, width);
        const int rank = __popcll(peers & lt_mask);
        // every lane of a digit group reads the counter before its lowest
        // lane advances it (LDS operations of a wavefront complete in order)
        const int32_t seen = wave_off[wave][dg];
        if (valid && rank == 0) wave_off[wave][dg] = seen + __popcll(peers);
        rk[r] = seen + rank;
    }
    __syncthreads();
    // the tile position of each wavefront's first item of a digit
#pragma unroll
    for (int q = 0; q < kPer; ++q) {
        int32_t acc = start[q];
#pragma unroll
        for (int w = 0; w < kWaves; ++w) {
            const int32_t c = wave_off[w][t * kPer + q];
            wave_off[w][t * kPer + q] = acc;
            acc += c;
        }
    }
    __syncthreads();
#pragma unroll
    for (int r = 0; r < ITEMS; ++r) {
        if (kk[r] < 0) continue;
        const int dg = (kk[r] >> shift) & (nb - 1);
        const int lpos = wave_off[wave][dg] + rk[r];
        if (lpos >= 0 && lpos < kTile) {  // always true for consistent counts
            lkey[lpos] = kk[r];
            lval[lpos] = vv[r];
        }
    }
    __syncthreads();
    for (int j = t; j < nvalid; j += kThreads) {
        const int32_t key = lkey[j];
        const int dg = (key >> shift) & (nb - 1);
        const int64_t pos = int64_t(delta[dg]) + j;
        if (pos >= 0 && pos < n) {  // always true for consistent counts
            keys_out[pos] = key;
            vals_out[pos] = lval[j];
        }
    }
}

// Reorder: scratch[j] = bunch[perm[j]] (7 columns + mask); the apply's deposit reads
// scratch and its kick writes it back to the bunch storage.
__global__ __launch_bounds__(kThreads) void k_gather_particles(
    const double* __restrict__ parts, int64_t stride, const uint8_t* __restrict__ masks,
    const int32_t* __restrict__ perm, int64_t n, double* __restrict__ scratch,
    uint8_t* __restrict__ smask, const DomainRec* dom)
{
    if (dom->error) return;
    for (int64_t j = int64_t(part_block()) * kThreads + threadIdx.x; j < n;
         j += int64_t(gridDim.x) * kThreads) {
        int64_t src = perm[j];
        if (src < 0 || src >= n) src = j;  // perm is a permutation of [0, n)
#pragma unroll
        for (int c = 0; c < 7; ++c) scratch[j + c * n] = parts[src + c * stride];
        smask[j] = masks[src];
    }
}

// The reorder of a storage in unknown order (an operator's first apply, on a
// bunch as it was populated or loaded): k_gather_particles then reads eight
// lines per particle from all over the bunch.  Here the particles first become
// records of the seven columns, read and written in order, and the reorder reads one record per particle and writes the columns
// of the storage itself: 1e6 particles in random order 141 -> 61 us, 4e6 625 ->
// 291, 1.6e7 2600 -> 1220 (with the kick's copy back of the gather).  In a
// storage already sorted the gather is the better one (its reads are in order).
constexpr int kRecordWords = 7;

__global__ __launch_bounds__(kThreads) void k_pack_records(
    const double* __restrict__ parts, int64_t stride, const uint8_t* __restrict__ masks, int64_t n,
    double* __restrict__ records, uint8_t* __restrict__ smask, const DomainRec* dom)
{
    if (dom->error) return;
    const int64_t i = int64_t(part_block()) * kThreads + threadIdx.x;
    if (i >= n) return;
    const uint8_t m = masks[i];
    double v[kRecordWords];
#pragma unroll
    for (int c = 0; c < kRecordWords; ++c) v[c] = parts[i + c * stride];
#pragma unroll
    for (int c = 0; c < kRecordWords; ++c) records[i * kRecordWords + c] = v[c];
    smask[i] = m;
}

__global__ __launch_bounds__(kThreads) void k_unpack_records(
    const double* __restrict__ records, const uint8_t* __restrict__ smask,
    const int32_t* __restrict__ perm, int64_t n, double* __restrict__ parts, int64_t stride,
    uint8_t* __restrict__ masks, const DomainRec* dom)
{
    if (dom->error) return;
    const int64_t j = int64_t(part_block()) * kThreads + threadIdx.x;
    if (j >= n) return;
    int64_t src = perm[j];
    if (src < 0 || src >= n) src = j;  // perm is a permutation of [0, n)
    double v[kRecordWords];
#pragma unroll
    for (int c = 0; c < kRecordWords; ++c) v[c] = records[src * kRecordWords + c];
    const uint8_t m = smask[src];
#pragma unroll
    for (int c = 0; c < kRecordWords; ++c) parts[j + c * stride] = v[c];
    masks[j] = m;
}

template <typename R>
__global__ void k_fill(R* __restrict__ p, int64_t n, R v)
{
    for (int64_t i = blockIdx.x * int64_t(blockDim.x) + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * blockDim.x)
        p[i] = v;
}

// ---------------------------------------------------------------------------
// CIC deposit (sv_zyx_rho_reducer_non_periodic, deposit.cc:309-395, launched
// :588-629): 8 corners with weights w0*aox*aoy*aoz (left to right), a corner
// written only if 0 < idx < g-1 in all three axes (ingrid, :21-30).
// Target: the G octant of rho2 (zyx, gx fastest).
//
// Precision form (FP32 grid): the cell index and offsets come from the FP64
// coordinates as above and the weights are unit charge weights aox*aoy*aoz;
// the physical weight w0 and the unit-peak scale return in FP64 at the kick.
// ---------------------------------------------------------------------------

// Deposit in windows of the bunch storage through an LDS node tile.  The
// storage is cell-sorted at every reorder (sort_period applies) and
// particles move a few cells per step, so consecutive slots stay a compact
// group of cells; PERM (storage never reordered): consecutive entries of this
// apply's sort permutation.  A block takes one window of 256 PER slots, each
// thread PER consecutive ones; the block reduces the window's cell bounding box, clears
// that box of nodes in LDS (up to kTileNodes FP64 nodes), and every particle
// adds its eight corner weights there with LDS FP64 atomics -- the corners of
// a thread's consecutive particles in one cell summed in registers first,
// the corner order permuted by lane so that the lanes of one cell hit eight
// different nodes at a time.  The block then adds the box's non-zero
// interior nodes to rho with global atomics (no sort, no scan, no run list).
// A window whose box does not fit gives each wavefront a quarter of the
// tile for the box of its own particles (no block barrier: LDS
// operations of one wavefront complete in order); a wavefront whose box does
// not fit either sums its corners in a direct-mapped FP64 cache of nodes in
// its quarter (a crowded node of a scattered storage then takes one add per
// wavefront), the rest going to rho directly.  Those wide
// windows lie at the two ends of the cell order (the tails of the bunch), so
// the block order is rotated to start the last eighth of the windows
// first and keep them off the end of the kernel.  Tile and grid accumulate in
// FP64 for both precisions; the precision form's unit weights are rounded to
// FP32 once per node and window, as they leave the tile, and their sum once
// more, by k_rho_round: FP64 holds the sums of FP32 values exactly, so the
// order of the global adds does not matter.  (Added in FP32 it left a node an
// error of up to 6e-8 per window; over a few steps that moved single particles
// across a cell face, and so the slots of the next reorder, from one run to the
// next.)
// Measured against the windowed kernel it replaces (LDS radix sort of each
// window, lane runs, DPP segmented scan, LDS run list; PMC: 465 VALU
// instructions per particle), deposit phase per step over sort periods of
// 12: 96.1 -> 54.9 us at 4e6 particles FP64 (64x64x128), 333.5 -> 214.7 us
// at 1.6e7 FP32 (128x128x256).  Variants measured on the way (us at 4e6,
// over a sort period): one particle per lane-stride instead of four
// consecutive per thread 81-99; tiles of 2048 / 3072 nodes 93-105 / 83-93;
// 512-thread blocks (6144 / 8192 nodes) 61-102 / 60-75; without the
// per-wavefront fallback and the block-order rotation 68-78; the corner sums
// picked by an indexed load (through scratch) 107-134.  In the library
// (deposit phase per step, 4e6 FP64 / 1.6e7 FP32): 4080 nodes (32 KiB with
// the box, 5 blocks per CU) 56.5 / 224.7 against 55.7 / 215.5; the same at 5
// waves per SIMD (96 VGPRs, 32 bytes spilled) 60.0 / 228.8; 3060 nodes at 6
// waves 93.3 / 351.9; the last eighth rotated first 55.8 / 215.7; 2 or 8
// slots per thread (windows of 512 / 2048) 61.6 / 242.4 and 72.6 / 287.0
// against 54.8 / 215.3.  With brick-ordered keys, sort period 24: the last
// eighth / sixteenth / thirty-second rotated first, or none, 54.6-54.8 /
// 55.4-55.5 / 54.3-54.5 / 56.1-56.3 at 4e6 and 200.6-200.7 / 201.3-202.4 /
// 201.8-202.3 / 203.5 at 1.6e7; 3 slots per thread 57.4-57.6 / 212.2-212.5.
// Weights formed in the lane's corner order, offsets once per thread and the
// flush's divisions by multiplication (248 -> 176 VALU instructions per
// particle): 46.9 -> 42.3 us per launch at 4e6 FP64, 226 -> 218 at 1.6e7 FP32
// (about four runs a thread late in the sort period; then the LDS atomics and
// the four blocks a CU holds are the limit).  The thread's slots loaded
// together, two a load, instead of one after the other behind a bounds branch
// each: 48.1 -> 43.5 us and 217 -> 206 (right after a sort 41 -> 35.4 and 144 ->
// 119); 4080 nodes with a fifth block per CU 43.8 and 206.
constexpr int kTileThreads = 256;
constexpr int kTileNodes = 4096;                        // FP64 nodes of the LDS tile (32 KiB)
constexpr int kTileTailDiv = 8;                         // 1/8 of the windows rotated first
constexpr int kTileWaves = kTileThreads / 64;

// Wavefront min / max, the same value in every lane: prefix reductions
// inside each row of 16 lanes by DPP moves (a lane with no source keeps its
// own value), then the four row results read from lanes 15, 31, 47, 63.
// Every lane of the wavefront calls it.  (Measured against six ds_bpermute
// exchanges per value, brick-ordered keys, sort period 24, deposit / kick
// phase: 54.3-54.7 / 64.4-64.7 -> 51.9-52.2 / 61.8-62.1 us at 4e6 FP64,
// 200.6-200.9 / 237.4-238.3 -> 190.2-190.8 / 233.5-233.8 us at 1.6e7 FP32.)
__device__ __forceinline__ int wave_min(int v)
{
    v = min(v, dpp_move<kDppRowShr + 1>(v, v));
    v = min(v, dpp_move<kDppRowShr + 2>(v, v));
    v = min(v, dpp_move<kDppRowShr + 4>(v, v));
    v = min(v, dpp_move<kDppRowShr + 8>(v, v));
    return min(min(__builtin_amdgcn_readlane(v, 15), __builtin_amdgcn_readlane(v, 31)),
               min(__builtin_amdgcn_readlane(v, 47), __builtin_amdgcn_readlane(v, 63)));
}
__device__ __forceinline__ int wave_max(int v)
{
    v = max(v, dpp_move<kDppRowShr + 1>(v, v));
    v = max(v, dpp_move<kDppRowShr + 2>(v, v));
    v = max(v, dpp_move<kDppRowShr + 4>(v, v));
    v = max(v, dpp_move<kDppRowShr + 8>(v, v));
    return max(max(__builtin_amdgcn_readlane(v, 15), __builtin_amdgcn_readlane(v, 31)),
               max(__builtin_amdgcn_readlane(v, 47), __builtin_amdgcn_readlane(v, 63)));
}

// Corners in this lane's order: position k is corner k ^ (lane mod 8) (x bit
// 0, y bit 1, z bit 2), so that the lanes of one cell add to eight different
// nodes at a time.  The order enters where the three factor pairs are formed,
// so weights and run sums come out in it and nothing is permuted afterwards
// (permuting the sums by register swaps at every run took 48 instructions).
struct LaneCorners {
    bool sx, sy, sz;
    __device__ __forceinline__ explicit LaneCorners(int lane)
        : sx(lane & 1), sy(lane & 2), sz(lane & 4) {}
    // weights in the reference's order of products, w0*wx*wy*wz left to right
    // (deposit.cc:366-391)
    __device__ __forceinline__ void weights(double w0, double ox, double oy, double oz,
                                            double (&w)[8]) const
    {
        const double aox = 1.0 - ox, aoy = 1.0 - oy, aoz = 1.0 - oz;
        const double fx[2] = {sx ? ox : aox, sx ? aox : ox};
        const double fy[2] = {sy ? oy : aoy, sy ? aoy : oy};
        const double fz[2] = {sz ? oz : aoz, sz ? aoz : oz};
#pragma unroll
        for (int k = 0; k < 8; ++k) w[k] = w0 * fx[k & 1] * fy[(k >> 1) & 1] * fz[k >> 2];
    }
    // node offsets in a box of nx x ny x .. nodes
    __device__ __forceinline__ void offsets(int nx, int ny, int (&off)[8]) const
    {
        const int px[2] = {sx ? 1 : 0, sx ? 0 : 1};
        const int py[2] = {sy ? nx : 0, sy ? 0 : nx};
        const int pz[2] = {sz ? nx * ny : 0, sz ? 0 : nx * ny};
#pragma unroll
        for (int k = 0; k < 8; ++k) off[k] = px[k & 1] + py[(k >> 1) & 1] + pz[k >> 2];
    }
};

// This thread's particles into a tile whose box starts at (bx, by, bz):
// consecutive particles of one cell summed first.
template <int PER>
__device__ __forceinline__ void tile_deposit(double* tile, int bx, int by, int bz, int nx, int ny,
                                             const LaneCorners& lc, double w0,
                                             const int (&ix)[PER], const int (&iy)[PER],
                                             const int (&iz)[PER], const bool (&ok)[PER],
                                             const double (&ox)[PER], const double (&oy)[PER],
                                             const double (&oz)[PER])
{
    int off[8];
    lc.offsets(nx, ny, off);
    double s[8];
    int cur = -1;
    auto add = [&] {
#pragma unroll
        for (int k = 0; k < 8; ++k) unsafeAtomicAdd(&tile[cur + off[k]], s[k]);
    };
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        if (!ok[q]) continue;
        const int b0 = ((iz[q] - bz) * ny + (iy[q] - by)) * nx + (ix[q] - bx);
        double w[8];
        lc.weights(w0, ox[q], oy[q], oz[q], w);
        if (b0 == cur) {
#pragma unroll
            for (int k = 0; k < 8; ++k) s[k] += w[k];
        } else {
            if (cur >= 0) add();
#pragma unroll
            for (int k = 0; k < 8; ++k) s[k] = w[k];
            cur = b0;
        }
    }
    if (cur >= 0) add();
}

// What the window adds to a node.
template <bool UNIT> __device__ __forceinline__ double grid_sum(double v)
{
    return UNIT ? double(float(v)) : v;
}

// The non-zero interior nodes of a tile (box at (bx, by, bz), nx x ny x ..,
// `nodes` in all) into rho, node e of the thread's share first..step.
template <bool UNIT>
__device__ __forceinline__ void tile_flush(const double* tile, int nodes, int first, int step,
                                           int bx, int by, int bz, int nx, int ny, int gx, int gy,
                                           int gz, double* __restrict__ rho)
{
    const uint32_t mx = small_magic(nx), my = small_magic(ny);
    for (int e = first; e < nodes; e += step) {
        const double v = tile[e];
        if (v == 0.0) continue;
        const int r = small_div(e, mx), rz = small_div(r, my);
        const int cx = bx + e - r * nx, cy = by + r - rz * ny, cz = bz + rz;
        if (cx > 0 && cx < gx - 1 && cy > 0 && cy < gy - 1 && cz > 0 && cz < gz - 1)
            unsafeAtomicAdd(rho + (int64_t(cz) * gy + cy) * gx + cx, grid_sum<UNIT>(v));
    }
}

// PER consecutive doubles from p (8-byte aligned), two a load.
template <int PER>
__device__ __forceinline__ void load_run(const double* __restrict__ p, double (&v)[PER])
{
    typedef double pair __attribute__((ext_vector_type(2), aligned(8)));
#pragma unroll
    for (int q = 0; q + 1 < PER; q += 2) {
        const pair t = *reinterpret_cast<const pair*>(p + q);
        v[q] = t.x;
        v[q + 1] = t.y;
    }
}

// UNIT (precision form): unit weights; w0 and the unit-peak scale return at
// the kick.
template <bool UNIT, int PER, bool PERM>
__global__ __launch_bounds__(kTileThreads) void k_deposit_tile(
    const double* __restrict__ parts, int64_t stride, const uint8_t* __restrict__ masks,
    const int32_t* __restrict__ perm, int64_t n, int gx, int gy, int gz,
    const DomainRec* __restrict__ dom, double* __restrict__ rho)
{
    __shared__ double tile[kTileNodes];
    __shared__ int box[kTileWaves][6];
    if (dom->error) return;
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const LaneCorners lc(lane);
    const double lx = dom->left[0], ly = dom->left[1], lz = dom->left[2];
    const double ihx = dom->inv_h[0], ihy = dom->inv_h[1], ihz = dom->inv_h[2];
    const double w0 = UNIT ? 1.0 : dom->w0;
    // the last eighth of the windows (one tail of the bunch) first
    const int nb = int(gridDim.x), tail = nb / kTileTailDiv;
    const int blk = (int(blockIdx.x) + nb - tail) % nb;
    const int64_t base = int64_t(blk) * (kTileThreads * PER) + int64_t(t) * PER;
    // every load of the thread's slots in flight together, 16 bytes at a time
    // (a column starts anywhere: 8-byte alignment); a slot past n reads the last
    double x[PER], y[PER], z[PER];
    uint8_t m[PER];
    if (!PERM && PER > 1 && (int64_t(blk) + 1) * (kTileThreads * PER) <= n) {
        load_run<PER>(parts + base, x);
        load_run<PER>(parts + base + 2 * stride, y);
        load_run<PER>(parts + base + 4 * stride, z);
#pragma unroll
        for (int q = 0; q < PER; ++q) m[q] = masks[base + q];
    } else {
#pragma unroll
        for (int q = 0; q < PER; ++q) {
            const int64_t j = min(base + q, n - 1);
            uint8_t active;
            if (PERM) {
                const Packed p = reinterpret_cast<const Packed*>(parts)[perm[j]];
                x[q] = p.x;
                y[q] = p.y;
                z[q] = p.z;
                active = p.active != 0.0;
            } else {
                x[q] = parts[j];
                y[q] = parts[j + 2 * stride];
                z[q] = parts[j + 4 * stride];
                active = masks[j];
            }
            m[q] = base + q < n ? active : uint8_t(0);
        }
    }
    int ix[PER], iy[PER], iz[PER];
    double ox[PER], oy[PER], oz[PER];
    bool ok[PER];
    int lo[3] = {INT32_MAX, INT32_MAX, INT32_MAX}, hi[3] = {-1, -1, -1};
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        // a particle outside [0, g-2] in any axis has no interior corner
        const bool in_x = grid_cell(x[q], lx, ihx, gx, ix[q], ox[q]);
        const bool in_y = grid_cell(y[q], ly, ihy, gy, iy[q], oy[q]);
        const bool in_z = grid_cell(z[q], lz, ihz, gz, iz[q], oz[q]);
        ok[q] = in_x & in_y & in_z & (m[q] != 0);
        lo[0] = min(lo[0], ok[q] ? ix[q] : INT32_MAX); hi[0] = max(hi[0], ok[q] ? ix[q] : -1);
        lo[1] = min(lo[1], ok[q] ? iy[q] : INT32_MAX); hi[1] = max(hi[1], ok[q] ? iy[q] : -1);
        lo[2] = min(lo[2], ok[q] ? iz[q] : INT32_MAX); hi[2] = max(hi[2], ok[q] ? iz[q] : -1);
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        lo[a] = wave_min(lo[a]);
        hi[a] = wave_max(hi[a]);
    }
    if (lane == 0)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            box[wave][a] = lo[a];
            box[wave][3 + a] = hi[a];
        }
    __syncthreads();
    int blo[3], bhi[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        blo[a] = box[0][a];
        bhi[a] = box[0][3 + a];
#pragma unroll
        for (int w = 1; w < kTileWaves; ++w) {
            blo[a] = min(blo[a], box[w][a]);
            bhi[a] = max(bhi[a], box[w][3 + a]);
        }
    }
    if (bhi[0] < 0) return;  // nothing of the window on the grid (block-uniform)
    // the box of cells lo..hi has (hi - lo + 2) nodes per axis
    const int nx = bhi[0] - blo[0] + 2, ny = bhi[1] - blo[1] + 2, nz = bhi[2] - blo[2] + 2;
    const int nodes = nx * ny * nz;
    if (nodes <= kTileNodes) {  // block-uniform
        for (int e = t; e < nodes; e += kTileThreads) tile[e] = 0.0;
        __syncthreads();
        tile_deposit(tile, blo[0], blo[1], blo[2], nx, ny, lc, w0, ix, iy, iz, ok, ox, oy, oz);
        __syncthreads();
        tile_flush<UNIT>(tile, nodes, t, kTileThreads, blo[0], blo[1], blo[2], nx, ny, gx, gy, gz,
                         rho);
        return;
    }
    // the window's box does not fit: this wavefront's own box in its quarter
    constexpr int kWaveNodes = kTileNodes / kTileWaves;
    double* wtile = tile + wave * kWaveNodes;
    const int wnx = hi[0] - lo[0] + 2, wny = hi[1] - lo[1] + 2, wnz = hi[2] - lo[2] + 2;
    const int wn = wnx * wny * wnz;
    if (hi[0] >= 0 && wn <= kWaveNodes) {  // wavefront-uniform; no block barrier below
        for (int e = lane; e < wn; e += 64) wtile[e] = 0.0;
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        tile_deposit(wtile, lo[0], lo[1], lo[2], wnx, wny, lc, w0, ix, iy, iz, ok, ox, oy, oz);
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
        __builtin_amdgcn_wave_barrier();
        tile_flush<UNIT>(wtile, wn, lane, 64, lo[0], lo[1], lo[2], wnx, wny, gx, gy, gz, rho);
        return;
    }
    // scattered particles (the sparse tails, or a storage out of cell order):
    // the quarter becomes a direct-mapped cache of kCacheSlots nodes (key =
    // node index, claimed by compare-and-swap) summed in FP64; a corner whose
    // slot holds another node goes to rho directly
    constexpr int kCacheSlots = kWaveNodes / 2;
    double* cval = wtile;
    int* ckey = reinterpret_cast<int*>(wtile + kCacheSlots);
    for (int e = lane; e < kCacheSlots; e += 64) {
        cval[e] = 0.0;
        ckey[e] = -1;
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        if (!ok[q]) continue;
        double w[8];
        LaneCorners(0).weights(w0, ox[q], oy[q], oz[q], w);
#pragma unroll
        for (int c = 0; c < 8; ++c) {
            const int cx = ix[q] + (c & 1), cy = iy[q] + ((c >> 1) & 1), cz = iz[q] + (c >> 2);
            if (!(cx > 0 && cx < gx - 1 && cy > 0 && cy < gy - 1 && cz > 0 && cz < gz - 1))
                continue;
            const int node = (cz * gy + cy) * gx + cx;
            const int slot = int((uint32_t(node) * 2654435761u) >> 23) & (kCacheSlots - 1);
            const int held = atomicCAS(&ckey[slot], -1, node);
            if (held == -1 || held == node)
                unsafeAtomicAdd(&cval[slot], w[c]);
            else
                unsafeAtomicAdd(rho + node, grid_sum<UNIT>(w[c]));
        }
    }
    __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "wavefront");
    __builtin_amdgcn_wave_barrier();
    for (int e = lane; e < kCacheSlots; e += 64) {
        const int node = ckey[e];
        if (node >= 0) unsafeAtomicAdd(rho + node, grid_sum<UNIT>(cval[e]));
    }
}

// The precision form's density: the FP64 sums of unit weights rounded to FP32,
// and the peak of that (all entries >= 0, so the IEEE bit patterns order like
// the values): block max (wavefront butterflies, then LDS), one integer
// atomicMax per block into the domain record (cleared by k_domain_finish each
// apply); the grid is bounded so few atomics meet, about 10 ns each on their
// one address (128x128x256, up to 256 / 512 / 1024 / 2048 blocks of 16, 8, 8 and
// 8 loads per round: 11.4 / 13.3 / 17.7 / 28.2 us; the peak alone, of FP32 sums,
// took 8.7).
__global__ __launch_bounds__(kThreads) void k_rho_round(const double* __restrict__ sums,
                                                        float* __restrict__ rho, int64_t G,
                                                        DomainRec* __restrict__ dom)
{
    __shared__ float wmax[kThreads / 64];
    if (dom->error) return;
    float m = 0.0f;
    // sixteen independent loads in flight per lane and round
    const int64_t T = int64_t(gridDim.x) * kThreads;
    int64_t i = blockIdx.x * int64_t(kThreads) + threadIdx.x;
    for (; i + 15 * T < G; i += 16 * T) {
        double v[16];
#pragma unroll
        for (int u = 0; u < 16; ++u) v[u] = sums[i + u * T];
#pragma unroll
        for (int u = 0; u < 16; ++u) {
            const float r = float(v[u]);
            rho[i + u * T] = r;
            m = fmaxf(m, r);
        }
    }
    for (; i < G; i += T) {
        const float r = float(sums[i]);
        rho[i] = r;
        m = fmaxf(m, r);
    }
    m = __int_as_float(wave_max(__float_as_int(m)));  // m >= 0: the bits order like the values
    if ((threadIdx.x & 63) == 0) wmax[threadIdx.x >> 6] = m;
    __syncthreads();
    if (threadIdx.x == 0) {
        float b = wmax[0];
        for (int w = 1; w < kThreads / 64; ++w) b = fmaxf(b, wmax[w]);
        if (b > 0.0f) atomicMax(&dom->rho_peak, __float_as_int(b));
    }
}

// ---------------------------------------------------------------------------
// E field (zyx::alg_force_extractor_doubled_domain, space_charge_3d_kernels.h:
// 217-307): E = -(phi[+1] - phi[-1]) * (0.5/h) on interior nodes, 0 on the
// boundary.  Stored interleaved (Ex, Ey, Ez, 0) per node for the kick's
// gathers.
// ---------------------------------------------------------------------------
template <typename R>
__global__ __launch_bounds__(kThreads) void k_efield(const R* __restrict__ phi, int gx, int gy,
                                                     int gz, const DomainRec* __restrict__ dom,
                                                     typename vec4<R>::type* __restrict__ E)
{
    if (dom->error) return;
    const double ihx = dom->half_inv_h[0], ihy = dom->half_inv_h[1], ihz = dom->half_inv_h[2];
    const int64_t G = int64_t(gx) * gy * gz;
    for (int64_t i = blockIdx.x * int64_t(kThreads) + threadIdx.x; i < G;
         i += int64_t(gridDim.x) * kThreads) {
        int ix = int(i % gx);
        int64_t r = i / gx;
        int iy = int(r % gy), iz = int(r / gy);
        typename vec4<R>::type e;
        e.x = R(0); e.y = R(0); e.z = R(0); e.w = R(0);
        if (!(ix == 0 || ix == gx - 1 || iy == 0 || iy == gy - 1 || iz == 0 || iz == gz - 1)) {
            const int64_t sy = gx, sz = int64_t(gx) * gy;
            e.x = R(-(double(phi[i + 1]) - double(phi[i - 1])) * ihx);
            e.y = R(-(double(phi[i + sy]) - double(phi[i - sy])) * ihy);
            e.z = R(-(double(phi[i + sz]) - double(phi[i - sz])) * ihz);
        }
        E[i] = e;
    }
}

// ---------------------------------------------------------------------------
// Kick (zyx::alg_kicker, space_charge_3d_kernels.h:91-215): kicked iff
// 0 <= idx < g-1 in all axes; trilinear Ez -> energy kick on dp/p, then Ey
// -> y', then Ex -> x', each interpolation summed in the reference's corner
// order.  Momenta accumulate in FP64 for every precision.
// k_kick also applies the map program that follows the kick in the
// split-operator sequence to every active particle in the same pass (one read
// and one write of the six coordinates for kick + maps); SCHED: the served
// form's scheduled program instead of the one passed by value.
// COPY (the apply that reordered the bunch): the particles are read from the
// cell-sorted copy the reorder gathered (src: 7 columns of stride n, and its
// masks), and every particle's 7 columns and mask are written to the bunch
// storage -- the reorder's copy back, folded into the kick.
// ---------------------------------------------------------------------------
// Kick factor: the FP64 form's is the record's; the precision form's grid
// holds unit-weight charge scaled to unit peak, so w0 * peak returns here.
template <typename R>
__device__ __forceinline__ double kick_factor(const DomainRec& d)
{
    if (sizeof(R) == sizeof(double)) return d.factor;
    const float peak = __int_as_float(d.rho_peak);
    return d.factor * d.w0 * (peak > 0.0f ? double(peak) : 1.0);
}

// The momentum kick of one particle from the interpolated field (vx, vy, vz).
// The three square roots and the division by the uniform pref (rpref its
// correctly rounded reciprocal) take the short forms of sc3d_exact.h where
// the two differences are in their range -- always but for a particle almost
// at rest -- with the bits of the plain expressions below.
__device__ __forceinline__ void kick_momenta(double vx, double vy, double vz, double factor,
                                             double pref, double rpref, double m, double& xp,
                                             double& yp, double& dpop)
{
    const double p = pref + dpop * pref;
    const double ei2 = p * p + m * m;
    const double work = factor * (-pref) * vz;
    const double ei = sqrt_normal(ei2);
    const double ef = ei + work;
    const double pf2 = ef * ef - m * m, pi2 = ei * ei - m * m;
    if (fmin(pf2, pi2) > 1.0e-200 && fmax(pf2, pi2) < 1.0e200 && pref > 1.0e-100 &&
        pref < 1.0e100) {
        dpop += div_by(sqrt_normal(pf2) - sqrt_normal(pi2), pref, rpref);
    } else {
        const double Eoc_i = sqrt(ei2);
        const double Eoc_f = Eoc_i + work;
        dpop += (sqrt(Eoc_f * Eoc_f - m * m) - sqrt(Eoc_i * Eoc_i - m * m)) / pref;
    }
    yp += factor * vy;
    xp += factor * vx;
}

// Trilinear interpolation in the reference's corner order (weights left to
// right as there; fused multiply-adds for the sums).
template <typename R>
__device__ __forceinline__ void interpolate(const R (&ex)[8], const R (&ey)[8], const R (&ez)[8],
                                            double ox, double oy, double oz, double& vx,
                                            double& vy, double& vz)
{
    const double aox = 1.0 - ox, aoy = 1.0 - oy, aoz = 1.0 - oz;
    const double w[8] = {aoz * aoy * aox, aoz * aoy * ox, aoz * oy * aox, aoz * oy * ox,
                         oz * aoy * aox,  oz * aoy * ox,  oz * oy * aox,  oz * oy * ox};
    vz = w[0] * double(ez[0]);
    vy = w[0] * double(ey[0]);
    vx = w[0] * double(ex[0]);
#pragma unroll
    for (int c = 1; c < 8; ++c) {
        vz = __builtin_fma(w[c], double(ez[c]), vz);
        vy = __builtin_fma(w[c], double(ey[c]), vy);
        vx = __builtin_fma(w[c], double(ex[c]), vx);
    }
}

template <typename R, bool COPY, bool SCHED>
__global__ __launch_bounds__(kThreads, 4) void k_kick(double* __restrict__ parts, int64_t stride,
                                                   uint8_t* __restrict__ masks, int64_t n,
                                                   int gx, int gy, int gz,
                                                   const DomainRec* __restrict__ dom,
                                                   const typename vec4<R>::type* __restrict__ E,
                                                   double pref, double rpref, double m,
                                                   MapProgram prog, Sched sc, const double* __restrict__ src,
                                                   const uint8_t* __restrict__ smasks)
{
    if (dom->error) return;
    const MapProgram* __restrict__ sp = SCHED ? sc.progs + sc.ctl->after_prog : nullptr;
    const double lx = dom->left[0], ly = dom->left[1], lz = dom->left[2];
    const double ihx = dom->inv_h[0], ihy = dom->inv_h[1], ihz = dom->inv_h[2];
    const double factor = kick_factor<R>(*dom);
    const double* __restrict__ rd = COPY ? src : parts;
    const int64_t rs = COPY ? n : stride;
    const int64_t i = blockIdx.x * int64_t(kThreads) + threadIdx.x;
    if (i >= n) return;
    // the mask and all six coordinates in flight together (fused kick of the
    // tracked cell, 4e6 particles: 180.9 -> 178.5 us)
    const uint8_t on = COPY ? smasks[i] : masks[i];
    double x = rd[i], y = rd[i + 2 * rs], cdt = rd[i + 4 * rs];
    double xp = rd[i + rs], yp = rd[i + 3 * rs], dpop = rd[i + 5 * rs];
    if (!COPY) {
        asm volatile("" ::"v"(x), "v"(y), "v"(cdt), "v"(xp), "v"(yp), "v"(dpop));
        if (!on) return;
    }
    double ox, oy, oz;
    int ix, iy, iz;
    bool in = grid_cell(x, lx, ihx, gx, ix, ox);
    in = grid_cell(y, ly, ihy, gy, iy, oy) && in;
    in = grid_cell(cdt, lz, ihz, gz, iz, oz) && in && on;
    if (COPY) {
        masks[i] = on;
        parts[i + 6 * stride] = rd[i + 6 * rs];
    }
    if (in) {
        const int64_t b0 = (int64_t(iz) * gy + iy) * gx + ix;
        const int64_t b1 = b0 + int64_t(gx) * gy;
        const int64_t c[8] = {b0, b0 + 1, b0 + gx, b0 + gx + 1, b1, b1 + 1, b1 + gx, b1 + gx + 1};
        R ex[8], ey[8], ez[8];
#pragma unroll
        for (int k = 0; k < 8; ++k) {
            const auto v = E[c[k]];
            ex[k] = v.x;
            ey[k] = v.y;
            ez[k] = v.z;
        }
        double vx, vy, vz;
        interpolate<R>(ex, ey, ez, ox, oy, oz, vx, vy, vz);
        kick_momenta(vx, vy, vz, factor, pref, rpref, m, xp, yp, dpop);
    }
    if (on) {
        const double xp0 = xp, yp0 = yp;
        auto again = [&] {
            const int64_t j = reread_index(i);
            x = rd[j];
            y = rd[j + 2 * rs];
            cdt = rd[j + 4 * rs];
            xp = xp0;
            yp = yp0;
        };
        if (SCHED)
            apply_program(*sp, x, xp, y, yp, cdt, dpop, again);
        else
            apply_program(prog, x, xp, y, yp, cdt, dpop, again);
    }
    parts[i] = x;
    parts[i + 2 * stride] = y;
    parts[i + 4 * stride] = cdt;
    parts[i + stride] = xp;
    parts[i + 3 * stride] = yp;
    parts[i + 5 * stride] = dpop;
}

// The kick without maps over windows of the bunch storage (PER
// particles per lane, lane-interleaved so every load is coalesced) with the
// field of each window's box of nodes staged in LDS: the storage is
// cell-sorted at every reorder, so a window's particles share few nodes, and
// the eight-corner gathers read LDS instead of going through the vector
// cache (a timing probe without the gathers ran the kick in 47 of its 72 us
// at 4e6 particles on 64x64x128).  A window whose box exceeds the tile (the
// sparse tails, a storage out of cell order) gathers from global memory as
// k_kick does.  Same arithmetic in the same order as k_kick: the tile holds
// copies of the field values.  Measured (kick us, 4e6 FP64 on 64x64x128 /
// 1.6e7 FP32 on 128x128x256, one run): k_kick 75.7 / 242; 2 particles per
// lane and 1024 nodes 69.4 / 224; 4 and 2048 nodes 70.5 / 240; 1 and 512
// nodes 73.9 / 234.  With the maps fused (k_kick) the extra
// registers of the tile version cost more than the gathers save: the fused
// kick stays on k_kick.  With the short square roots and division, fused
// multiply-adds in the interpolation and the cheaper cell test (391 -> 310
// VALU instructions per particle): 61.0 -> 58.5 / 247 -> 233 us per launch,
// 73 bytes per particle at 5.0 TB/s; k_kick with one drift fused 75.7 -> 69.7.
// All of a lane's loads in flight together, no branch between them: 58.3 ->
// 54.2 / 234.6 -> 226.8 us.
constexpr int kKickNodes = 1024;

template <typename R, bool COPY, int PER>
__global__ __launch_bounds__(kThreads) void k_kick_tile(
    double* __restrict__ parts, int64_t stride, uint8_t* __restrict__ masks, int64_t n, int gx,
    int gy, int gz, const DomainRec* __restrict__ dom, const typename vec4<R>::type* __restrict__ E,
    double pref, double rpref, double m, const double* __restrict__ src,
    const uint8_t* __restrict__ smasks)
{
    __shared__ R tile[3][kKickNodes];
    __shared__ int box[kThreads / 64][6];
    if (dom->error) return;
    const double lx = dom->left[0], ly = dom->left[1], lz = dom->left[2];
    const double ihx = dom->inv_h[0], ihy = dom->inv_h[1], ihz = dom->inv_h[2];
    const double factor = kick_factor<R>(*dom);
    const int t = threadIdx.x, lane = t & 63, wave = t >> 6;
    const int64_t base = int64_t(blockIdx.x) * (kThreads * PER) + t;
    const double* __restrict__ rd = COPY ? src : parts;
    const int64_t rs = COPY ? n : stride;
    double x[PER], y[PER], cdt[PER], xp[PER], yp[PER], dpop[PER];
    double ox[PER], oy[PER], oz[PER];
    int ix[PER], iy[PER], iz[PER];
    double id[PER];  // COPY only
    uint8_t on[PER];
    bool in[PER];
    int lo[3] = {INT32_MAX, INT32_MAX, INT32_MAX}, hi[3] = {-1, -1, -1};
    // every load in flight together; a lane past n reads the last particle
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int64_t i = min(base + int64_t(q) * kThreads, n - 1);
        on[q] = COPY ? smasks[i] : masks[i];
        x[q] = rd[i];
        y[q] = rd[i + 2 * rs];
        cdt[q] = rd[i + 4 * rs];
        xp[q] = rd[i + rs];
        yp[q] = rd[i + 3 * rs];
        dpop[q] = rd[i + 5 * rs];
        if (COPY) id[q] = rd[i + 6 * rs];
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        const int64_t i = base + int64_t(q) * kThreads;
        if (COPY && i < n) {
            masks[i] = on[q];
            parts[i] = x[q];
            parts[i + 2 * stride] = y[q];
            parts[i + 4 * stride] = cdt[q];
            parts[i + 6 * stride] = id[q];
        }
        const bool in_x = grid_cell(x[q], lx, ihx, gx, ix[q], ox[q]);
        const bool in_y = grid_cell(y[q], ly, ihy, gy, iy[q], oy[q]);
        const bool in_z = grid_cell(cdt[q], lz, ihz, gz, iz[q], oz[q]);
        in[q] = in_x & in_y & in_z & (on[q] != 0) & (i < n);
        lo[0] = min(lo[0], in[q] ? ix[q] : INT32_MAX); hi[0] = max(hi[0], in[q] ? ix[q] : -1);
        lo[1] = min(lo[1], in[q] ? iy[q] : INT32_MAX); hi[1] = max(hi[1], in[q] ? iy[q] : -1);
        lo[2] = min(lo[2], in[q] ? iz[q] : INT32_MAX); hi[2] = max(hi[2], in[q] ? iz[q] : -1);
    }
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        lo[a] = wave_min(lo[a]);
        hi[a] = wave_max(hi[a]);
    }
    if (lane == 0)
#pragma unroll
        for (int a = 0; a < 3; ++a) {
            box[wave][a] = lo[a];
            box[wave][3 + a] = hi[a];
        }
    __syncthreads();
    int blo[3], bhi[3];
#pragma unroll
    for (int a = 0; a < 3; ++a) {
        blo[a] = box[0][a];
        bhi[a] = box[0][3 + a];
#pragma unroll
        for (int w = 1; w < kThreads / 64; ++w) {
            blo[a] = min(blo[a], box[w][a]);
            bhi[a] = max(bhi[a], box[w][3 + a]);
        }
    }
    // the box of cells lo..hi has (hi - lo + 2) nodes per axis
    const int nx = bhi[0] - blo[0] + 2, ny = bhi[1] - blo[1] + 2, nz = bhi[2] - blo[2] + 2;
    const bool staged = bhi[0] >= 0 && nx * ny * nz <= kKickNodes;  // block-uniform
    if (staged) {
        const int nodes = nx * ny * nz;
        const uint32_t mx = small_magic(nx), my = small_magic(ny);
        for (int e = t; e < nodes; e += kThreads) {
            const int r = small_div(e, mx), cx = e - r * nx;
            const int cz = small_div(r, my), cy = r - cz * ny;
            const auto v = E[(int64_t(blo[2] + cz) * gy + blo[1] + cy) * gx + blo[0] + cx];
            tile[0][e] = v.x;
            tile[1][e] = v.y;
            tile[2][e] = v.z;
        }
        __syncthreads();
    }
#pragma unroll
    for (int q = 0; q < PER; ++q) {
        if (COPY ? base + int64_t(q) * kThreads >= n : !in[q]) continue;
        if (in[q]) {
            R ex[8], ey[8], ez[8];
            if (staged) {
                const int b0 = ((iz[q] - blo[2]) * ny + iy[q] - blo[1]) * nx + ix[q] - blo[0];
                const int b1 = b0 + nx * ny;
                const int c[8] = {b0, b0 + 1, b0 + nx, b0 + nx + 1,
                                  b1, b1 + 1, b1 + nx, b1 + nx + 1};
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    ex[k] = tile[0][c[k]];
                    ey[k] = tile[1][c[k]];
                    ez[k] = tile[2][c[k]];
                }
            } else {
                const int64_t b0 = (int64_t(iz[q]) * gy + iy[q]) * gx + ix[q];
                const int64_t b1 = b0 + int64_t(gx) * gy;
                const int64_t c[8] = {b0, b0 + 1, b0 + gx, b0 + gx + 1,
                                      b1, b1 + 1, b1 + gx, b1 + gx + 1};
#pragma unroll
                for (int k = 0; k < 8; ++k) {
                    const auto v = E[c[k]];
                    ex[k] = v.x;
                    ey[k] = v.y;
                    ez[k] = v.z;
                }
            }
            double vx, vy, vz;
            interpolate<R>(ex, ey, ez, ox[q], oy[q], oz[q], vx, vy, vz);
            kick_momenta(vx, vy, vz, factor, pref, rpref, m, xp[q], yp[q], dpop[q]);
        }
        const int64_t i = base + int64_t(q) * kThreads;
        parts[i + stride] = xp[q];
        parts[i + 3 * stride] = yp[q];
        parts[i + 5 * stride] = dpop[q];
    }
}

// ---------------------------------------------------------------------------
// Populate: Philox-4x32-10 (Salmon et al., SC'11) keyed by the 64-bit seed,
// counter (id_lo, id_hi, call, 0); 53-bit uniforms in (0,1); Box-Muller.
// ---------------------------------------------------------------------------
__device__ __forceinline__ uint4 philox4x32_10(uint4 c, uint2 k)
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        uint32_t hi0 = __umulhi(0xD2511F53u, c.x), lo0 = 0xD2511F53u * c.x;
        uint32_t hi1 = __umulhi(0xCD9E8D57u, c.z), lo1 = 0xCD9E8D57u * c.z;
        c = make_uint4(hi1 ^ c.y ^ k.x, lo1, hi0 ^ c.w ^ k.y, lo0);
        k.x += 0x9E3779B9u;
        k.y += 0xBB67AE85u;
    }
    return c;
}

// (m + 0.5) 2^-53 for the top 53 bits m of (a, b): in (0, 1]; exactly 1.0
// only for m = 2^53 - 1 (the sum rounds up), which the transforms below take.
__device__ __forceinline__ double u53(uint32_t a, uint32_t b)
{
    uint64_t m = (uint64_t(a) << 21) | (b >> 11);
    return (double(m) + 0.5) * 0x1.0p-53;
}

// Box-Muller's log and sin/cos(2 pi u) from IEEE basic operations only
// (+ - * / sqrt floor frexp, no FMA contraction in this library), so the
// same seed gives the same bunch bit for bit on any IEEE machine, whatever
// its libm.  Accuracy (measured against 200-bit arithmetic over 2e5 samples):
// log within 0.76 ulp, sin and cos within 2 ulp.
//
// log(u), u in (0, 1]: u = m 2^e with m in [sqrt(1/2), sqrt(2)), f = m - 1
// (exact), s = f / (2 + f), log(1 + f) = 2 atanh(s) = f - (f^2/2 - s (f^2/2
// + R)) with R = sum_k 2 s^2k / (2k+1), k = 1..11 (|s| <= 0.1716, the
// truncation is below 1e-18 relative) -- the arrangement of fdlibm's e_log.c
// with Taylor coefficients; ln 2 split into a 32-bit head (e * head exact)
// and its tail.
__device__ __forceinline__ double det_log(double u)
{
    constexpr double kLn2Hi = 0x1.62e42feep-1;             // ln 2, top 32 bits
    constexpr double kLn2Lo = 0x1.a39ef35793c76p-33;       // ln 2 - kLn2Hi
    constexpr double kSqrtHalf = 0x1.6a09e667f3bcdp-1;
    int e;
    double m = frexp(u, &e);
    if (m < kSqrtHalf) {
        m = m + m;
        e = e - 1;
    }
    const double f = m - 1.0;
    const double s = f / (2.0 + f);
    const double z = s * s;
    double R = 2.0 / 23.0;
    R = 2.0 / 21.0 + z * R;
    R = 2.0 / 19.0 + z * R;
    R = 2.0 / 17.0 + z * R;
    R = 2.0 / 15.0 + z * R;
    R = 2.0 / 13.0 + z * R;
    R = 2.0 / 11.0 + z * R;
    R = 2.0 / 9.0 + z * R;
    R = 2.0 / 7.0 + z * R;
    R = 2.0 / 5.0 + z * R;
    R = 2.0 / 3.0 + z * R;
    R = z * R;
    const double hfsq = 0.5 * f * f;
    const double dk = double(e);
    return dk * kLn2Hi + (f - (hfsq - (s * (hfsq + R) + dk * kLn2Lo)));
}

// sin and cos of 2 pi u, u in (0, 1]: quadrant q = floor(4u), r = 4u - q
// (both exact), the angle folded to a = r or 1 - r <= 1/2 (exact), x = a pi/2
// <= pi/4 (one rounding), Taylor series of sin x to x^19 and cos x to x^20
// (truncation below 1e-19), then the exact quadrant rotation.
__device__ __forceinline__ void det_sincos2pi(double u, double* sn, double* cs)
{
    constexpr double kPi2 = 0x1.921fb54442d18p+0;  // pi / 2
    const double t = 4.0 * u;
    const double q = floor(t);
    const double r = t - q;
    const bool fold = r > 0.5;
    const double a = fold ? 1.0 - r : r;
    const double x = a * kPi2;
    const double z = x * x;
    double S = -1.0 / 121645100408832000.0;  // -1/19!
    S = 1.0 / 355687428096000.0 + z * S;     // 1/17!
    S = -1.0 / 1307674368000.0 + z * S;      // -1/15!
    S = 1.0 / 6227020800.0 + z * S;          // 1/13!
    S = -1.0 / 39916800.0 + z * S;           // -1/11!
    S = 1.0 / 362880.0 + z * S;              // 1/9!
    S = -1.0 / 5040.0 + z * S;               // -1/7!
    S = 1.0 / 120.0 + z * S;                 // 1/5!
    S = -1.0 / 6.0 + z * S;                  // -1/3!
    const double s0 = x + x * (z * S);
    double Cp = 1.0 / 2432902008176640000.0;  // 1/20!
    Cp = -1.0 / 6402373705728000.0 + z * Cp;  // -1/18!
    Cp = 1.0 / 20922789888000.0 + z * Cp;     // 1/16!
    Cp = -1.0 / 87178291200.0 + z * Cp;       // -1/14!
    Cp = 1.0 / 479001600.0 + z * Cp;          // 1/12!
    Cp = -1.0 / 3628800.0 + z * Cp;           // -1/10!
    Cp = 1.0 / 40320.0 + z * Cp;              // 1/8!
    Cp = -1.0 / 720.0 + z * Cp;               // -1/6!
    Cp = 1.0 / 24.0 + z * Cp;                 // 1/4!
    Cp = -1.0 / 2.0 + z * Cp;                 // -1/2!
    const double c0 = 1.0 + z * Cp;
    const double sq = fold ? c0 : s0;  // sin and cos of the angle in the quadrant
    const double cq = fold ? s0 : c0;
    switch (int(q) & 3) {
    case 0: *sn = sq; *cs = cq; break;
    case 1: *sn = cq; *cs = -sq; break;
    case 2: *sn = -sq; *cs = -cq; break;
    default: *sn = -cq; *cs = sq; break;
    }
}

__global__ __launch_bounds__(kThreads) void k_populate(double* __restrict__ parts, int64_t stride,
                                                       int64_t n, uint8_t* __restrict__ masks,
                                                       PopulateArgs a)
{
    for (int64_t i = blockIdx.x * int64_t(kThreads) + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * kThreads) {
        int64_t id = a.id0 + i;
        uint2 key = make_uint2(uint32_t(a.seed), uint32_t(a.seed >> 32));
        double u[6];
        for (int call = 0; call < 3; ++call) {
            uint4 r = philox4x32_10(
                make_uint4(uint32_t(id), uint32_t(uint64_t(id) >> 32), uint32_t(call), 0u), key);
            u[2 * call] = u53(r.x, r.y);
            u[2 * call + 1] = u53(r.z, r.w);
        }
        double g[6];
        for (int k = 0; k < 3; ++k) {
            double rad = sqrt(-2.0 * det_log(u[2 * k]));
            double s, c;
            det_sincos2pi(u[2 * k + 1], &s, &c);
            g[2 * k] = rad * c;
            g[2 * k + 1] = rad * s;
        }
        for (int r = 0; r < 6; ++r) {
            double v = a.mean[r];
            for (int c = 0; c <= r; ++c) v += a.chol[r * (r + 1) / 2 + c] * g[c];
            parts[i + r * stride] = v;
        }
        parts[i + 6 * stride] = double(id);
        masks[i] = 1;
    }
}

// ---------------------------------------------------------------------------
// host launchers
// ---------------------------------------------------------------------------
// Blocks for n items, at most cap, rounded up to a multiple of 8 (the
// XCD-contiguous block order of part_block needs one; the kernels launched
// on these grids let surplus blocks run empty).
static int grid_for(int64_t n, int cap = 8192)
{
    int64_t b = (n + kThreads - 1) / kThreads;
    if (b < 1) b = 1;
    if (b > cap) b = cap;
    return int((b + 7) / 8 * 8);
}

static unsigned round8(int64_t b) { return unsigned((b + 7) / 8 * 8); }

void launch_tail_counts(const double* parts, int64_t stride, const uint8_t* masks, int64_t n,
                        const TailArgs& a, unsigned long long* counts, hipStream_t st)
{
    uint32_t* partial = reinterpret_cast<uint32_t*>(counts + 8);
    const int blocks = n > 0 ? grid_for(n, kTailBlocks) : 0;
    if (blocks > 0)
        hipLaunchKernelGGL(k_tail_counts, dim3(blocks), dim3(kThreads), 0, st, parts, stride,
                           masks, n, a, partial);
    hipLaunchKernelGGL(k_tail_finish, dim3(6), dim3(kThreads), 0, st, partial, blocks, counts);
}


__global__ __launch_bounds__(kThreads) void k_adjust(double* __restrict__ parts, int64_t stride,
                                                     int64_t n, AdjustArgs a)
{
    for (int64_t i = blockIdx.x * int64_t(kThreads) + threadIdx.x; i < n;
         i += int64_t(gridDim.x) * kThreads) {
        double d[6], o[6];
#pragma unroll
        for (int k = 0; k < 6; ++k) d[k] = parts[i + k * stride] - a.mean[k];
#pragma unroll
        for (int j = 0; j < 6; ++j) {
            double s = 0.0;
#pragma unroll
            for (int k = 0; k < 6; ++k) s += d[k] * a.A[j * 6 + k];
            o[j] = s + a.means[j];
        }
#pragma unroll
        for (int j = 0; j < 6; ++j) parts[i + j * stride] = o[j];
    }
}

void launch_adjust(double* parts, int64_t stride, int64_t n, const AdjustArgs& a, hipStream_t st)
{
    if (n > 0)
        hipLaunchKernelGGL(k_adjust, dim3(grid_for(n)), dim3(kThreads), 0, st, parts, stride, n,
                           a);
}

// The density grid (grid_bytes, a multiple of 16) is cleared here: by the
// chunk pass when its chunks are enough for slices of at most 32 KiB each,
// else by a fill of its own.
void launch_domain(const double* parts, int64_t stride, const uint8_t* masks, int64_t n,
                   double* P, const DomainFinishArgs& a, DomainRec* dom, const Sched& sc,
                   void* grid, int64_t grid_bytes, hipStream_t st)
{
    const int64_t nch = (n + 4095) / 4096;
    const int64_t grid16 = grid_bytes / 16;
    const bool chunks = !a.fixed && nch > 0;
    const bool clear = chunks && grid_bytes <= nch * 32768;
    if (chunks)
        hipLaunchKernelGGL(k_domain_partial, dim3(unsigned(nch)), dim3(kThreads), 0, st, parts,
                           stride, masks, n, P, sc.ctl, static_cast<uint4*>(grid),
                           clear ? grid16 : int64_t(0));
    if (!clear)
        hipLaunchKernelGGL(k_fill<uint4>, dim3(grid_for(grid16, 2048)), dim3(kThreads), 0, st,
                           static_cast<uint4*>(grid), grid16, make_uint4(0, 0, 0, 0));
    hipLaunchKernelGGL(k_domain_finish, dim3(1), dim3(kThreads), 0, st, P, chunks ? nch : 0, a,
                       dom, sc);
}

void launch_step_begin(StepCtl* ctl, hipStream_t st)
{
    hipLaunchKernelGGL(k_step_begin, dim3(1), dim3(64), 0, st, ctl);
}

template <int ITEMS, int WIDTH>
static void launch_sort_tiles(const double* parts, int64_t stride, const uint8_t* masks, int64_t n,
                              int gx, int gy, int gz, const DomainRec* dom, SortBuffers& b,
                              int bits, Packed* packed, hipStream_t st)
{
    static_assert(kThreads * ITEMS * (2048 >> WIDTH) >= kSortTileItems, "counts buffer");
    constexpr int kTile = kThreads * ITEMS;
    const int nblk = int((n + kTile - 1) / kTile);
    const int passes = (bits + WIDTH - 1) / WIDTH;
    const int width = (bits + passes - 1) / passes;
    const int nb = 1 << width;
    const dim3 grid(round8(nblk)), block(kThreads);
    const int32_t* kin = b.keys0;
    const int32_t* vin = nullptr;
    int32_t* kout[2] = {b.keysA, b.keysB};
    int32_t* vout[2] = {b.valsA, b.valsB};
    for (int p = 0; p < passes; ++p) {
        const int shift = width * p;
        if (p == 0)
            hipLaunchKernelGGL((k_radix_count<true, ITEMS, WIDTH>), grid, block, 0, st, parts,
                               stride, masks, gx, gy, gz, b.keys0, n, shift, width, b.counts, nblk,
                               dom, packed);
        else
            hipLaunchKernelGGL((k_radix_count<false, ITEMS, WIDTH>), grid, block, 0, st,
                               (const double*)nullptr, int64_t(0), (const uint8_t*)nullptr, gx,
                               gy, gz, const_cast<int32_t*>(kin), n, shift, width, b.counts,
                               nblk, dom, (Packed*)nullptr);
        hipLaunchKernelGGL(k_radix_scan, dim3(nb), block, 0, st, b.counts, nblk, b.totals, dom);
        hipLaunchKernelGGL((k_radix_scatter<ITEMS, WIDTH>), grid, block, 0, st, kin, vin, n, shift,
                           width, b.counts, b.totals, nblk, kout[p & 1], vout[p & 1], dom);
        kin = kout[p & 1];
        vin = vout[p & 1];
    }
    b.perm = const_cast<int32_t*>(vin);
}

void launch_sort(const double* parts, int64_t stride, const uint8_t* masks, int64_t n, int gx,
                 int gy, int gz, const DomainRec* dom, SortBuffers& b, double* packed,
                 hipStream_t st)
{
    const int64_t G = int64_t(gx) * gy * gz;
    int bits = 0;
    while ((int64_t(1) << bits) <= G) ++bits;  // keys in [0, G]
    auto go = [&](auto f) { f(parts, stride, masks, n, gx, gy, gz, dom, b, bits, reinterpret_cast<Packed*>(packed), st); };
    // Tile: small enough to fill the chip, large enough for the scan of the
    // tiles' counts.  Whole sort with tiles of 1024 / 2048 / 4096 items, us:
    // 1e5 particles 37 / 47 / 69, 1e6 56 / 62 / 80, 2e6 79 / 80 / 94, 4e6 125 /
    // 116 / 120, 1.6e7 589 / 430 / 395 (4096 and one load per round before: 98
    // at 1e5, 123 at 2e6).  Digits of 9 bits where they take fewer passes, with
    // the small tiles: 1e5 particles on 32x32x64, 2 passes 30, 3 passes 37; of
    // 10 bits they gain nothing (2e6 on 64x64x64: 85 against 80).
    if (n <= 2500000) {
        if ((bits + kWideDigitBits - 1) / kWideDigitBits < (bits + kMaxDigitBits - 1) / kMaxDigitBits)
            go(launch_sort_tiles<4, kWideDigitBits>);
        else
            go(launch_sort_tiles<4, kMaxDigitBits>);
    } else if (n <= 8000000) {
        go(launch_sort_tiles<8, kMaxDigitBits>);
    } else {
        go(launch_sort_tiles<16, kMaxDigitBits>);
    }
}

void launch_reorder(double* parts, int64_t stride, uint8_t* masks, int64_t n, const int32_t* perm,
                    double* scratch, uint8_t* smask, const DomainRec* dom, hipStream_t st)
{
    // One particle per thread up to 1.7e7 particles: the gather is bound by the latency of its
    // random reads, so more waves in flight help (measured at 1.6e7 particles, one sort every
    // 12 steps: sort plus reorder 132 us per step on average with 65536 blocks, 138 with 8192).
    // The copy of the gathered bunch back into the storage is the kick's (k_kick*<.., COPY>):
    // until then the deposit reads the gathered copy.
    const dim3 grid(grid_for(n, 65536));
    hipLaunchKernelGGL(k_gather_particles, grid, dim3(kThreads), 0, st, parts, stride, masks,
                       perm, n, scratch, smask, dom);
}

void launch_reorder_records(double* parts, int64_t stride, uint8_t* masks, int64_t n,
                            const int32_t* perm, double* scratch, uint8_t* smask,
                            const DomainRec* dom, hipStream_t st)
{
    const dim3 grid(round8((n + kThreads - 1) / kThreads));
    hipLaunchKernelGGL(k_pack_records, grid, dim3(kThreads), 0, st, parts, stride, masks, n,
                       scratch, smask, dom);
    hipLaunchKernelGGL(k_unpack_records, grid, dim3(kThreads), 0, st, scratch, smask, perm, n,
                       parts, stride, masks, dom);
}

template <bool UNIT>
static void launch_deposit_tiles(const double* parts, int64_t stride, const uint8_t* masks,
                                 const int32_t* perm, int64_t n, int gx, int gy, int gz,
                                 DomainRec* dom, double* rho, bool served, hipStream_t st)
{
    auto launch = [&](auto kernel, int per) {
        const int64_t win = kTileThreads * int64_t(per), nb = (n + win - 1) / win;
        if (nb < 1) return;
        hipLaunchKernelGGL(kernel, dim3(unsigned(nb)), dim3(kTileThreads), 0, st, parts, stride,
                           masks, perm, n, gx, gy, gz, dom, rho);
    };
    // Slots per thread: fewer where the windows would leave CUs idle (deposit
    // phase at 1 / 2 / 4 slots, us: 1e4 particles 8.6 / 9.8 / 14.9, 1e5 8.4 / 9.1
    // / 11.6 on 32x32x64; 4e5 on 64x64x128 14.8 / 12.6 / 15.5; 1e6 23.4 / 20.6 /
    // 19.9); one through a permutation, whose random reads want the wavefronts
    // (1e5 11.1 / 12.4 / 18.0, 1e6 25.2 / 25.8 / 31.6, 4e6 82.8 / 81.8 / 84.1).
    // The precision form's windows are the groups that are rounded together, and
    // smaller ones move a sparse bunch's field by more than the results of four
    // slots ever differed among themselves (n < 60000: dp/p by 1e-8 where they
    // differ by 2e-9), so an operator's applies keep four.  A server's, whose
    // jobs' results are emittances and moments (1e-9), take the same rule as
    // FP64 (128 mixed jobs: 3.29 -> 3.22 s).
    if (perm != nullptr)
        launch(k_deposit_tile<UNIT, 1, true>, 1);
    else if (UNIT && !served)
        launch(k_deposit_tile<UNIT, 4, false>, 4);
    else if (n < 250000)
        launch(k_deposit_tile<UNIT, 1, false>, 1);
    else if (n < 750000)
        launch(k_deposit_tile<UNIT, 2, false>, 2);
    else
        launch(k_deposit_tile<UNIT, 4, false>, 4);
}

void launch_deposit(const double* parts, int64_t stride, const uint8_t* masks,
                    const int32_t* perm, int64_t n, int gx, int gy, int gz, DomainRec* dom,
                    double* sums, float* rho32, bool served, hipStream_t st)
{
    if (!rho32) {
        launch_deposit_tiles<false>(parts, stride, masks, perm, n, gx, gy, gz, dom, sums, served,
                                    st);
        return;
    }
    launch_deposit_tiles<true>(parts, stride, masks, perm, n, gx, gy, gz, dom, sums, served, st);
    const int64_t G = int64_t(gx) * gy * gz;
    hipLaunchKernelGGL(k_rho_round, dim3(grid_for(G / 16, 256)), dim3(kThreads), 0, st, sums, rho32,
                       G, dom);
}

template <typename R>
void launch_efield(const R* phi, int gx, int gy, int gz, const DomainRec* dom,
                   typename vec4<R>::type* E, hipStream_t st)
{
    hipLaunchKernelGGL(k_efield<R>, dim3(grid_for(int64_t(gx) * gy * gz)), dim3(kThreads), 0, st,
                       phi, gx, gy, gz, dom, E);
}

template <typename R>
void launch_kick(double* parts, int64_t stride, uint8_t* masks, int64_t n, int gx, int gy, int gz,
                 const DomainRec* dom, const typename vec4<R>::type* E, double pref, double m,
                 const MapProgram& prog, const Sched& sc, const double* src,
                 const uint8_t* smasks, hipStream_t st)
{
    if (n <= 0) return;
    const bool copy = src != nullptr;
    if (prog.n == 0 && !sc.progs) {
        auto tiles = [&](auto kernel, int64_t win) {
            hipLaunchKernelGGL(kernel, dim3(unsigned((n + win - 1) / win)), dim3(kThreads), 0, st,
                               parts, stride, masks, n, gx, gy, gz, dom, E, pref, 1.0 / pref, m,
                               src, smasks);
        };
        // one particle per lane where two would leave CUs idle (kick us, 1 / 2
        // per lane: 1e4 particles 5.6 / 6.1, 1e6 20.4 / 20.8, 4e6 60.0 / 54.2)
        if (n < 1000000)
            copy ? tiles(k_kick_tile<R, true, 1>, kThreads)
                 : tiles(k_kick_tile<R, false, 1>, kThreads);
        else
            copy ? tiles(k_kick_tile<R, true, 2>, 2 * kThreads)
                 : tiles(k_kick_tile<R, false, 2>, 2 * kThreads);
        return;
    }
    const dim3 grid(unsigned((n + kThreads - 1) / kThreads));
    auto launch = [&](auto kernel) {
        hipLaunchKernelGGL(kernel, grid, dim3(kThreads), 0, st, parts, stride, masks, n, gx, gy,
                           gz, dom, E, pref, 1.0 / pref, m, prog, sc, src, smasks);
    };
    if (sc.progs)
        copy ? launch(k_kick<R, true, true>) : launch(k_kick<R, false, true>);
    else
        copy ? launch(k_kick<R, true, false>) : launch(k_kick<R, false, false>);
}

void launch_populate(double* parts, int64_t stride, int64_t n, uint8_t* masks,
                     const PopulateArgs& a, hipStream_t st)
{
    hipLaunchKernelGGL(k_populate, dim3(grid_for(n)), dim3(kThreads), 0, st, parts, stride, n,
                       masks, a);
}

template void launch_efield<double>(const double*, int, int, int, const DomainRec*, double4*,
                                    hipStream_t);
template void launch_efield<float>(const float*, int, int, int, const DomainRec*, float4*,
                                   hipStream_t);
template void launch_kick<double>(double*, int64_t, uint8_t*, int64_t, int, int, int,
                                  const DomainRec*, const double4*, double, double,
                                  const MapProgram&, const Sched&, const double*, const uint8_t*,
                                  hipStream_t);
template void launch_kick<float>(double*, int64_t, uint8_t*, int64_t, int, int, int,
                                 const DomainRec*, const float4*, double, double,
                                 const MapProgram&, const Sched&, const double*, const uint8_t*,
                                 hipStream_t);

}  // namespace sc3d
