// Multi-right-hand-side PCG: A X = B for up to 8 right-hand sides sharing one matrix, in one sequence of
// launches. The reference solves one system per call (SolverCG::solve, src/linear_algebra/
// linear_solver.cu:301-376); each column here follows that recurrence (Jacobi or no preconditioner,
// the same stopping test on (r, M^-1 r)) with its own scalars and its own convergence, so a column's
// iterates equal a single-RHS solve's up to the order of the dot-product reductions.
//
// Layout: the solver's work vectors are interleaved, v[i * G + j] = component i of column j, with G the
// column count rounded up to 1, 2, 4 or 8. A row is handled by a group of G consecutive lanes, lane j of
// the group taking column j: the group reads the row's values and column indices once (one broadcast
// load per entry for all columns) and gathers G contiguous values per column index, so the matrix stream
// is shared by the columns and the gathers are G-wide. Dot products are reduced per column in a fixed
// order (deterministic). The caller's X and B are column-major (column j at X + j * n).
//
// PFEM_PRECISION_MIXED: PCG with reliable updates (residual replacement). The iterations run on FP32
// vectors and the FP32 copy of A (half the bytes); the solution accumulates in FP64. When a column's
// recursive residual has fallen by a set factor (10x by default) since the last replacement, or passes
// the stopping test, the
// column spends one iteration slot on a replacement: x += x_s in FP64, r = b - A x with the FP64 matrix,
// the stopping test on that true residual, and the search direction continued from it (beta = new
// gamma / old gamma). Unlike restarted refinement, the Krylov recurrence is never restarted, so the
// iteration count stays close to the FP64 solver's, and convergence is decided on FP64 residuals.
#include <algorithm>
#include <cmath>
#include <cstddef>
#include <cstring>
#include <memory>
#include <vector>

#include "device.hpp"
#include "internal.hpp"
#include "solver.hpp"

namespace pfem {

constexpr int kMaxRhs = 8;
constexpr int kMBlock = 512;              // workgroup of the multi-RHS kernels: one wave per column when it adds up partials
constexpr int kMWaves = kMBlock / 64;
constexpr int kMGrid = 768;               // most workgroups of a kernel that leaves partial sums
constexpr int kMStream = 512;             // workgroups of the vector kernels
static_assert(kMGrid % 64 == 0 && kMStream <= kMGrid, "a wave adds up a series in whole rounds");

// One column's scalars. gam: gamma of the current residual; rzmax: gamma at the last replacement (mixed); mode:
// 0 iterating, 1 replacement due, 2 direction update after a replacement (mixed).
struct MCol {
    double gam, thr, res, alpha, beta, rzmax;
    int it, done, converged, nan, mode, nrep;
};

// Two of these take turns within an iteration: the kernel after the product reads the first and leaves the
// second, the direction update reads the second and leaves the first, so that no workgroup reads what
// another of its launch writes.
struct MState {
    double tol, drop;
    int tol_mode, maxit, ncol, all_done;
    MCol col[kMaxRhs];
};

// N consecutive columns of a row, loaded and stored at once
template <typename T, int N>
struct Columns {
    typedef T type __attribute__((ext_vector_type(N)));
};

// Columns that one lane of a product takes
template <int G>
constexpr int kCols = G < 2 ? G : 2;

// Per-column block sums of NV values: lane l holds the NC columns from (l % (G / NC)) * NC on. Reduced over the
// wave with shuffles that keep the columns, then over the waves in order; part[(i * G + j) * gridDim.x +
// blockIdx.x] = value i of column j.
template <int G, int NV, int NC>
__device__ __forceinline__ void group_partials(double (&v)[NV][NC], double* __restrict__ part)
{
    __shared__ double sh[NV][kMWaves][G];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
#pragma unroll
    for (int i = 0; i < NV; ++i)
#pragma unroll
        for (int c = 0; c < NC; ++c) {
#pragma unroll
            for (int off = 32; off >= G / NC; off >>= 1) v[i][c] += __shfl_down(v[i][c], off, 64);
            if (lane < G / NC) sh[i][wid][lane * NC + c] = v[i][c];
        }
    __syncthreads();
    if (threadIdx.x < G) {
#pragma unroll
        for (int i = 0; i < NV; ++i) {
            double s = sh[i][0][threadIdx.x];
            for (int w = 1; w < kMWaves; ++w) s += sh[i][w][threadIdx.x];
            part[((size_t)i * G + threadIdx.x) * gridDim.x + blockIdx.x] = s;
        }
    }
}

// Total of a partial series of nb <= kMGrid terms, valid in lane 0 of the wave. Every load is issued before
// the first addition (one memory round trip); lane t adds terms t, t + 64, ... in order, then wave_sum.
__device__ __forceinline__ double series_total(const double* __restrict__ part, int nb)
{
    constexpr int kPer = kMGrid / 64;
    const int lane = threadIdx.x & 63;
    double t[kPer];
#pragma unroll
    for (int u = 0; u < kPer; ++u) {
        const int k = lane + u * 64;
        t[u] = k < nb ? part[k] : 0.0;
    }
    double s = 0.0;
#pragma unroll
    for (int u = 0; u < kPer; ++u) s += t[u];
    return wave_sum(s);
}

// The scalar step between two kernels, at the head of the second one: wave j adds up column j's partials and
// moves the column's scalars on with f(column, total); every workgroup does so for itself (a few loads from
// L2, where a launch of one workgroup between the kernels took 8.5 to 12 us of a 78 us iteration of 8 columns
// x 0.27M rows), and workgroup 0 leaves the result in `out`. False if nothing is left to do.
template <int G, typename F>
__device__ __forceinline__ bool scalar_step(const MState* __restrict__ in, MState* __restrict__ out,
                                            const double* __restrict__ part, int nb, MCol (&sc)[G], F f)
{
    static_assert(G <= kMWaves, "one wave per column");
    const bool live = !in->all_done;
    const int wid = threadIdx.x >> 6;
    if (wid < G) {
        const double tot = live ? series_total(part + (size_t)wid * nb, nb) : 0.0;
        if ((threadIdx.x & 63) == 0) {
            MCol c = in->col[wid];
            if (live && !c.done) f(c, tot);
            sc[wid] = c;
        }
    }
    __syncthreads();
    if (blockIdx.x == 0) {
        if (threadIdx.x < G) out->col[threadIdx.x] = sc[threadIdx.x];
        if (threadIdx.x == 0) {
            int all = 1;
            for (int j = 0; j < G; ++j) all &= sc[j].done;
            out->all_done = all;
        }
    }
    return live;
}

// Elements o = i * G + j of the interleaved vectors in grid strides (a lane keeps its column), kMU at a time
constexpr int kMU = 4;
template <int G, typename F>
__device__ __forceinline__ void for_elements(int n, F f)
{
    const long m = (long)n * G, stride = (long)gridDim.x * kMBlock;
    for (long o = (long)blockIdx.x * kMBlock + threadIdx.x; o < m; o += kMU * stride) f(o, stride, m);
}

constexpr int kMTileNnz = 2048;   // non-zeros of a row tile staged in LDS
template <int G>
constexpr int tile_rows = kMBlock / G * kCols<G>;

// Row tiles of the multi-RHS products: tile t = rows [tiles[2t], tiles[2t+1]), at most tile_rows<G>
// rows and at most kMTileNnz non-zeros unless a single row is longer. A lane takes kCols columns of a row. Workgroup b takes a contiguous range of tiles; the
// ranges of XCD x (workgroups b = x mod 8) form the x-th band of rows, so neighbouring rows share their
// gathered vector entries in one L2. A tile's values, column indices and row offsets pass through registers into
// LDS with unit-stride loads that are in flight while the tile before is computed; each lane then adds
// val * x[col * G + j] over its rows left to right (the sequential order), with up to kU gathers per row in
// flight, and hands each sum to f(row, j, s). The lanes of a row gather G contiguous values.
// The gathers bound it (33M of them through L1 and L2, 8 columns x 0.27M rows): two columns to a lane halve the
// gather and LDS instructions, and six wavefronts a SIMD with four gathers in flight each hide more than four
// with eight or sixteen. 29.0 us before, with one column to a lane; now 22.2 (with eight in flight 24.5 at four
// wavefronts, 31.9 at six with spills; two in flight 24.3).
template <int G, typename T, typename VT, typename F>
__device__ __forceinline__ void for_tile_rows(int ntiles, const int* __restrict__ tiles, const int* __restrict__ rowptr,
                                              const int* __restrict__ col, const VT* __restrict__ val,
                                              const T* __restrict__ x, F f)
{
    constexpr int NC = kCols<G>, kLanes = G / NC;   // lanes per row
    constexpr int kTileRows = tile_rows<G>;
    using V = typename Columns<T, NC>::type;
    constexpr int kU = 4;
    constexpr int kStage = kMTileNnz / kMBlock;
    constexpr int kRp = (kTileRows + 1 + kMBlock - 1) / kMBlock;
    __shared__ __align__(16) VT sval[kMTileNnz];
    __shared__ int scol[kMTileNnz];
    __shared__ int rp[kTileRows + 1];
    const int nb = gridDim.x, b = blockIdx.x;
    const int rb = (b % 8) * (nb / 8) + b / 8;
    const int t0 = (int)((long)ntiles * rb / nb), t1 = (int)((long)ntiles * (rb + 1) / nb);
    const int j = threadIdx.x % kLanes * NC, q = threadIdx.x / kLanes;
    if (t0 >= t1) return;
    // bounds of tile t (current), of t + 1 (being staged) and of t + 2
    int r0 = tiles[2 * t0], r1 = tiles[2 * t0 + 1];
    int k0 = rowptr[r0], k1 = rowptr[r1];
    VT nv[kStage];
    int nc[kStage], nr[kRp];
    auto fetch = [&](int a, int z, int ka, int kz) {
#pragma unroll
        for (int u = 0; u < kRp; ++u) {
            const int i = threadIdx.x + u * kMBlock;
            nr[u] = i <= z - a ? rowptr[a + i] - ka : 0;
        }
        if (kz - ka <= kMTileNnz)
#pragma unroll
            for (int u = 0; u < kStage; ++u) {
                const int k = ka + (int)threadIdx.x + u * kMBlock;
                if (k < kz) {
                    nv[u] = val[k];
                    nc[u] = col[k];
                }
            }
    };
    fetch(r0, r1, k0, k1);
    int n0 = 0, n1 = 0, m0 = 0, m1 = 0;
    if (t0 + 1 < t1) {
        n0 = tiles[2 * t0 + 2];
        n1 = tiles[2 * t0 + 3];
        m0 = rowptr[n0];
        m1 = rowptr[n1];
    }
    for (int t = t0; t < t1; ++t) {
        const bool staged = k1 - k0 <= kMTileNnz;
        __syncthreads();   // the previous tile's readers are done with the LDS arrays
#pragma unroll
        for (int u = 0; u < kRp; ++u) {
            const int i = threadIdx.x + u * kMBlock;
            if (i <= r1 - r0) rp[i] = nr[u];
        }
        if (staged)
#pragma unroll
            for (int u = 0; u < kStage; ++u) {
                const int k = threadIdx.x + u * kMBlock;
                if (k < k1 - k0) {
                    sval[k] = nv[u];
                    scol[k] = nc[u];
                }
            }
        // the next tile is fetched while this one is computed
        if (t + 1 < t1) fetch(n0, n1, m0, m1);
        int p0 = 0, p1 = 0, l0 = 0, l1 = 0;
        if (t + 2 < t1) {
            p0 = tiles[2 * t + 4];
            p1 = tiles[2 * t + 5];
            l0 = rowptr[p0];
            l1 = rowptr[p1];
        }
        __syncthreads();
        const int row = r0 + q;
        if (staged) {
            if (row < r1) {
                V s = (V)(T)0;
                const int ka = rp[q], ke = rp[q + 1];
                for (int d = ka; d < ke; d += kU) {
                    V xv[kU];
                    T vv[kU];
#pragma unroll
                    for (int w = 0; w < kU; ++w)
                        if (d + w < ke) {
                            vv[w] = (T)sval[d + w];
                            xv[w] = *reinterpret_cast<const V*>(x + (size_t)scol[d + w] * G + j);
                        }
#pragma unroll
                    for (int w = 0; w < kU; ++w)
                        if (d + w < ke) s += vv[w] * xv[w];
                }
                f(row, j, s);
            }
        } else {
            // a row longer than a tile, on its own: all lanes form its products in LDS, the row's lanes add them in
            // order (3000 rows of 2800 entries: 1.90 -> 0.14 ms an iteration of 1 column, 2.24 -> 0.49 of 8, against a
            // lane or four that walked the row in memory)
            static_assert(sizeof(T) == sizeof(VT), "the products take the values' place");
            constexpr int kPart = kMTileNnz / G;
            T* const prod = reinterpret_cast<T*>(sval);
            V s = (V)(T)0;
            for (int d = k0; d < k1; d += kPart) {
                const int m = min(kPart, k1 - d);
#pragma unroll
                for (int u = 0; u < kStage; ++u) {
                    const int o = threadIdx.x + u * kMBlock;
                    if (o < m * G) prod[o] = (T)val[d + o / G] * x[(size_t)col[d + o / G] * G + o % G];
                }
                __syncthreads();
                if (q == 0)
#pragma unroll 8
                    for (int e = 0; e < m; ++e) s += *reinterpret_cast<const V*>(prod + e * G + j);
                __syncthreads();
            }
            if (q == 0) f(r0, j, s);
        }
        r0 = n0; r1 = n1; k0 = m0; k1 = m1;
        n0 = p0; n1 = p1; m0 = l0; m1 = l1;
    }
}

// ---- FP64 multi-RHS CG kernels
// r = b - A x, p = z = M^-1 r; partials (r, z) and (b, M^-1 b) per column
template <int G, bool JAC>
__global__ __launch_bounds__(kMBlock, 6) void k_m_init(int ntiles, const int* __restrict__ tiles,
                                                       const int* __restrict__ rowptr, const int* __restrict__ col,
                                                       const double* __restrict__ val, const double* __restrict__ x,
                                                       const double* __restrict__ b, const double* __restrict__ invd,
                                                       double* __restrict__ r, double* __restrict__ p, double* __restrict__ part)
{
    constexpr int NC = kCols<G>;
    using V = typename Columns<double, NC>::type;
    double v[2][NC] = {};
    for_tile_rows<G, double, double>(ntiles, tiles, rowptr, col, val, x, [&](int i, int j, V ax) {
        const size_t o = (size_t)i * G + j;
        const V bb = *reinterpret_cast<const V*>(b + o);
        const double d = JAC ? invd[i] : 1.0;
        const V rr = bb - ax;
        const V zz = JAC ? rr * d : rr;
        const V mb = JAC ? bb * d : bb;
        *reinterpret_cast<V*>(r + o) = rr;
        *reinterpret_cast<V*>(p + o) = zz;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            v[0][c] += rr[c] * zz[c];
            v[1][c] += bb[c] * mb[c];
        }
    });
    group_partials<G>(v, part);
}

// gamma_0, the per-column thresholds (linear_solver.cu:360; relative to (b, M^-1 b) on request, absolute
// for a zero column) and the columns already converged; one block
template <int G>
__global__ __launch_bounds__(kMBlock) void k_m_begin(MState* st, const double* __restrict__ part, int nb)
{
    __shared__ int done[G];
    const int j = threadIdx.x >> 6;
    if (j < G) {
        const double rz = series_total(part + (size_t)j * nb, nb), bmb = series_total(part + (size_t)(G + j) * nb, nb);
        if ((threadIdx.x & 63) == 0) {
            MCol c{};
            c.gam = c.rzmax = rz;
            c.thr = st->tol_mode == PFEM_TOL_RELATIVE && bmb > 0.0 ? st->tol * st->tol * bmb : st->tol * st->tol;
            c.nan = rz != rz;
            c.converged = rz < c.thr ? 1 : 0;
            c.done = j >= st->ncol || c.converged || c.nan;
            c.res = sqrt(fabs(rz));
            st->col[j] = c;
            done[j] = c.done;
        }
    }
    __syncthreads();
    if (threadIdx.x == 0) {
        int all = 1;
        for (int k = 0; k < G; ++k) all &= done[k];
        st->all_done = all;
    }
}

// q = A p; partials (p, q) per column
template <int G>
__global__ __launch_bounds__(kMBlock, 6) void k_m_spmv(int ntiles, const int* __restrict__ tiles,
                                                       const int* __restrict__ rowptr, const int* __restrict__ col,
                                                       const double* __restrict__ val, const double* __restrict__ p,
                                                       double* __restrict__ q, const MState* __restrict__ st,
                                                       double* __restrict__ part)
{
    if (st->all_done) return;
    constexpr int NC = kCols<G>;
    using V = typename Columns<double, NC>::type;
    double v[1][NC] = {};
    for_tile_rows<G, double, double>(ntiles, tiles, rowptr, col, val, p, [&](int i, int j, V ap) {
        const size_t o = (size_t)i * G + j;
        *reinterpret_cast<V*>(q + o) = ap;
        const V pp = *reinterpret_cast<const V*>(p + o);
#pragma unroll
        for (int c = 0; c < NC; ++c) v[0][c] += pp[c] * ap[c];
    });
    group_partials<G>(v, part);
}

// alpha = gamma / (p, q); r -= alpha q (updateXR, linear_solver.cu:68-77) for the active columns; partials
// (r, M^-1 r). x += alpha p is left to k_m_p, which reads p anyway: 8 vectors pass per iteration instead of 9.
template <int G, bool JAC>
__global__ __launch_bounds__(kMBlock) void k_m_update(int n, double* __restrict__ r, const double* __restrict__ q,
                                                      const double* __restrict__ invd, const MState* __restrict__ st,
                                                      MState* __restrict__ out, const double* __restrict__ pa, int na,
                                                      double* __restrict__ part)
{
    __shared__ MCol sc[G];
    const bool live = scalar_step<G>(st, out, pa, na, sc, [](MCol& c, double tot) { c.alpha = c.gam / tot; });
    if (!live) return;
    const int j = threadIdx.x % G;
    double v[1][1] = {};
    if (!sc[j].done) {
        const double alpha = sc[j].alpha;
        for_elements<G>(n, [&](long o, long stride, long m) {
            double rv[kMU], qv[kMU], dv[kMU];
#pragma unroll
            for (int u = 0; u < kMU; ++u) {
                const long k = o + u * stride;
                if (k < m) {
                    rv[u] = r[k];
                    qv[u] = q[k];
                    dv[u] = JAC ? invd[k / G] : 1.0;
                }
            }
#pragma unroll
            for (int u = 0; u < kMU; ++u) {
                const long k = o + u * stride;
                if (k < m) {
                    const double rr = rv[u] - alpha * qv[u];
                    r[k] = rr;
                    v[0][0] += rr * (JAC ? rr * dv[u] : rr);
                }
            }
        });
    }
    group_partials<G>(v, part);
}

// gamma_{k+1}, beta and the stopping test per active column; x += alpha p; p = M^-1 r + beta p (updateP,
// linear_solver.cu:79-87) for the columns still active
template <int G, bool JAC>
__global__ __launch_bounds__(kMBlock) void k_m_p(int n, double* __restrict__ x, double* __restrict__ p,
                                                 const double* __restrict__ r, const double* __restrict__ invd,
                                                 const MState* __restrict__ st, MState* __restrict__ out,
                                                 const double* __restrict__ pb, int nb)
{
    __shared__ MCol sc[G];
    __shared__ int was[G];
    const int maxit = st->maxit;
    if (threadIdx.x < G) was[threadIdx.x] = st->col[threadIdx.x].done;
    const bool live = scalar_step<G>(st, out, pb, nb, sc, [maxit](MCol& c, double gnew) {
        c.beta = gnew / c.gam;
        c.gam = gnew;
        c.it += 1;
        c.res = sqrt(fabs(gnew));
        if (gnew != gnew) {
            c.nan = 1;
            c.done = 1;
        } else if (gnew < c.thr) {
            c.converged = 1;
            c.done = 1;
        } else if (c.it >= maxit) {
            c.done = 1;
        }
    });
    if (!live) return;
    const int j = threadIdx.x % G;
    if (was[j]) return;
    const bool on = !sc[j].done;   // a column that stops here keeps its p: it is not used again
    const double alpha = sc[j].alpha, beta = sc[j].beta;
    for_elements<G>(n, [&](long o, long stride, long m) {
        double xv[kMU], pv[kMU], rv[kMU], dv[kMU];
#pragma unroll
        for (int u = 0; u < kMU; ++u) {
            const long k = o + u * stride;
            if (k < m) {
                xv[u] = x[k];
                pv[u] = p[k];
                rv[u] = r[k];
                dv[u] = JAC ? invd[k / G] : 1.0;
            }
        }
#pragma unroll
        for (int u = 0; u < kMU; ++u) {
            const long k = o + u * stride;
            if (k < m) {
                x[k] = xv[u] + alpha * pv[u];
                if (on) p[k] = (JAC ? rv[u] * dv[u] : rv[u]) + beta * pv[u];
            }
        }
    });
}

// ---- layout changes and refinement kernels
// column-major (column j at s + j * n, j < ncol) -> interleaved (columns ncol..G-1 zero)
template <int G, typename T>
__global__ void k_m_pack(int n, int ncol, const double* __restrict__ s, T* __restrict__ d)
{
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < (long)n * G; t += (long)gridDim.x * blockDim.x) {
        const int i = (int)(t / G), j = (int)(t % G);
        d[t] = j < ncol ? (T)s[(size_t)j * n + i] : (T)0;
    }
}

template <int G>
__global__ void k_m_unpack(int n, int ncol, const double* __restrict__ s, double* __restrict__ d)
{
    for (long t = (long)blockIdx.x * blockDim.x + threadIdx.x; t < (long)n * G; t += (long)gridDim.x * blockDim.x) {
        const int i = (int)(t / G), j = (int)(t % G);
        if (j < ncol) d[(size_t)j * n + i] = s[t];
    }
}

// ---- reliable-update PCG (PFEM_PRECISION_MIXED)
// r = b - A x (FP64), r_s = (float) r, p_s = D_s r_s, x_s = 0; partials (r, D r) and (b, D b) in FP64
template <int G, bool JAC>
__global__ __launch_bounds__(kMBlock, 6) void k_mr_init(int ntiles, const int* __restrict__ tiles, const int* __restrict__ rowptr,
                                                    const int* __restrict__ col, const double* __restrict__ val,
                                                    const double* __restrict__ x, const double* __restrict__ b,
                                                    const double* __restrict__ invd, const float* __restrict__ invd32,
                                                    float* __restrict__ rs, float* __restrict__ ps, float* __restrict__ xs,
                                                    double* __restrict__ part)
{
    constexpr int NC = kCols<G>;
    using V = typename Columns<double, NC>::type;
    using S = typename Columns<float, NC>::type;
    double v[2][NC] = {};
    for_tile_rows<G, double, double>(ntiles, tiles, rowptr, col, val, x, [&](int i, int j, V ax) {
        const size_t o = (size_t)i * G + j;
        const V bb = *reinterpret_cast<const V*>(b + o);
        const V rr = bb - ax;
        const double d = JAC ? invd[i] : 1.0;
        const float d32 = JAC ? invd32[i] : 1.0f;
        S r32;
#pragma unroll
        for (int c = 0; c < NC; ++c) {
            r32[c] = (float)rr[c];
            v[0][c] += rr[c] * (rr[c] * d);
            v[1][c] += bb[c] * (bb[c] * d);
        }
        *reinterpret_cast<S*>(rs + o) = r32;
        *reinterpret_cast<S*>(ps + o) = JAC ? r32 * d32 : r32;
        *reinterpret_cast<S*>(xs + o) = (S)0.0f;
    });
    group_partials<G>(v, part);
}

// Iterating columns: q_s = A_s p_s, partial (p_s, q_s). Columns due a replacement: r = b - A x with the
// FP64 matrix, r_s = (float) r, partial (r, D r). While some columns iterate and others are replaced both
// products pass over the rows, each keeping its own columns.
template <int G, bool JAC>
__global__ __launch_bounds__(kMBlock, 6) void k_mr_spmv(int ntiles, const int* __restrict__ tiles, const int* __restrict__ rowptr,
                                                    const int* __restrict__ col, const float* __restrict__ val32,
                                                    const double* __restrict__ val, const float* __restrict__ ps,
                                                    float* __restrict__ qs, const double* __restrict__ x,
                                                    const double* __restrict__ b, const double* __restrict__ invd,
                                                    float* __restrict__ rs, const MState* __restrict__ st,
                                                    double* __restrict__ part)
{
    if (st->all_done) return;
    constexpr int NC = kCols<G>;
    using V = typename Columns<double, NC>::type;
    using S = typename Columns<float, NC>::type;
    int rep = 0, iter = 0;   // columns, a bit each
    for (int c = 0; c < G; ++c)
        if (!st->col[c].done) (st->col[c].mode == 1 ? rep : iter) |= 1 << c;
    double v[1][NC] = {};
    if (iter)
        for_tile_rows<G, float, float>(ntiles, tiles, rowptr, col, val32, ps, [&](int i, int j, S ap) {
            const size_t o = (size_t)i * G + j;
            *reinterpret_cast<S*>(qs + o) = ap;
            const S pp = *reinterpret_cast<const S*>(ps + o);
#pragma unroll
            for (int c = 0; c < NC; ++c)
                if (!((rep >> (j + c)) & 1)) v[0][c] += (double)(pp[c] * ap[c]);
        });
    if (rep)
        for_tile_rows<G, double, double>(ntiles, tiles, rowptr, col, val, x, [&](int i, int j, V ax) {
            const size_t o = (size_t)i * G + j;
            const V bb = *reinterpret_cast<const V*>(b + o);
            const double d = JAC ? invd[i] : 1.0;
#pragma unroll
            for (int c = 0; c < NC; ++c)
                if ((rep >> (j + c)) & 1) {
                    const double rr = bb[c] - ax[c];
                    rs[o + c] = (float)rr;
                    v[0][c] += rr * (rr * d);
                }
        });
    group_partials<G>(v, part);
}

// Iterating columns: alpha = gamma / (p_s, q_s); r_s -= alpha q_s (FP32), partial (r_s, D_s r_s). A replaced
// column has its true gamma: the stopping test, then beta for the direction update.
template <int G, bool JAC>
__global__ __launch_bounds__(kMBlock) void k_mr_update(int n, float* __restrict__ rs, const float* __restrict__ qs,
                                                       const float* __restrict__ invd32, const MState* __restrict__ st,
                                                       MState* __restrict__ out, const double* __restrict__ pa, int na,
                                                       double* __restrict__ part)
{
    __shared__ MCol sc[G];
    const bool live = scalar_step<G>(st, out, pa, na, sc, [](MCol& c, double tot) {
        if (c.mode == 1) {
            c.nrep += 1;
            c.res = sqrt(fabs(tot));
            if (tot != tot) {
                c.nan = 1;
                c.done = 1;
            } else if (tot < c.thr) {
                c.converged = 1;
                c.done = 1;
            } else {
                c.beta = tot / c.gam;
                c.gam = c.rzmax = tot;
                c.mode = 2;
            }
        } else {
            c.mode = 0;
            c.alpha = c.gam / tot;
        }
    });
    if (!live) return;
    const int j = threadIdx.x % G;
    double v[1][1] = {};
    if (!sc[j].done && sc[j].mode == 0) {
        const float alpha = (float)sc[j].alpha;
        for_elements<G>(n, [&](long o, long stride, long m) {
            float rv[kMU], qv[kMU], dv[kMU];
#pragma unroll
            for (int u = 0; u < kMU; ++u) {
                const long k = o + u * stride;
                if (k < m) {
                    rv[u] = rs[k];
                    qv[u] = qs[k];
                    dv[u] = JAC ? invd32[k / G] : 1.0f;
                }
            }
#pragma unroll
            for (int u = 0; u < kMU; ++u) {
                const long k = o + u * stride;
                if (k < m) {
                    const float rr = rv[u] - alpha * qv[u];
                    rs[k] = rr;
                    v[0][0] += (double)(rr * (JAC ? rr * dv[u] : rr));
                }
            }
        });
    }
    group_partials<G>(v, part);
}

// gamma of the recursive residual: the iteration count, then either beta or a replacement (after a 10x
// drop since the last one, or when the recursive residual passes the stopping test). x_s += alpha p_s and
// p_s = D_s r_s + beta p_s (iterating columns; after a replacement the direction alone); a column due a
// replacement moves its correction into the FP64 solution: x += x_s, x_s = 0.
template <int G, bool JAC>
__global__ __launch_bounds__(kMBlock) void k_mr_p(int n, float* __restrict__ ps, const float* __restrict__ rs,
                                                  const float* __restrict__ invd32, double* __restrict__ x,
                                                  float* __restrict__ xs, const MState* __restrict__ st,
                                                  MState* __restrict__ out, const double* __restrict__ pb, int nb)
{
    __shared__ MCol sc[G];
    __shared__ int was[G];
    const int maxit = st->maxit;
    const double drop = st->drop;
    if (threadIdx.x < G) was[threadIdx.x] = st->col[threadIdx.x].done ? 2 : st->col[threadIdx.x].mode == 0;
    const bool live = scalar_step<G>(st, out, pb, nb, sc, [maxit, drop](MCol& c, double g) {
        if (c.mode != 0) return;
        c.it += 1;
        if (g != g) {
            c.nan = 1;
            c.done = 1;
        } else if (c.it >= maxit) {
            c.done = 1;
        } else if (g < c.thr || g < drop * c.rzmax) {
            c.mode = 1;
        } else {
            c.beta = g / c.gam;
            c.gam = g;
        }
    });
    if (!live) return;
    const int j = threadIdx.x % G;
    if (was[j] == 2) return;
    const bool step = was[j] == 1;                        // x_s moves
    const bool done = sc[j].done != 0, fold = !done && sc[j].mode == 1;
    const float alpha = (float)sc[j].alpha, beta = (float)sc[j].beta;
    for_elements<G>(n, [&](long o, long stride, long m) {
        float xv[kMU], pv[kMU], rv[kMU], dv[kMU];
#pragma unroll
        for (int u = 0; u < kMU; ++u) {
            const long k = o + u * stride;
            if (k < m) {
                xv[u] = step ? xs[k] : 0.0f;
                pv[u] = ps[k];
                rv[u] = rs[k];
                dv[u] = JAC ? invd32[k / G] : 1.0f;
            }
        }
#pragma unroll
        for (int u = 0; u < kMU; ++u) {
            const long k = o + u * stride;
            if (k < m) {
                const float xn = step ? xv[u] + alpha * pv[u] : 0.0f;
                if (fold) {
                    x[k] += (double)xn;
                    xs[k] = 0.0f;
                } else {
                    if (step) xs[k] = xn;
                    if (!done) ps[k] = (JAC ? rv[u] * dv[u] : rv[u]) + beta * pv[u];
                }
            }
        }
    });
}

// x += x_s over every column (a converged column's x_s is zero: its last replacement folded it in)
__global__ void k_mr_fold(long m, double* __restrict__ x, const float* __restrict__ xs)
{
    const long t = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (t < m) x[t] += (double)xs[t];
}

__global__ void k_m_to32(long n, float* __restrict__ d, const double* __restrict__ s)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = (float)s[i];
}

// ---- host side
struct MultiWork {
    int n = 0, G = 0, ncol = 0;
    std::shared_ptr<Pattern> pat;
    DevArray<int> tiles;                // row tiles of the products (for_tile_rows)
    int ntiles = 0;
    DevArray<double> x, b, r, p, q;    // FP64 interleaved (x, b also the refinement's solution and RHS)
    DevArray<float> x32, r32, p32, q32;  // reliable updates: x_s, r_s, p_s, q_s
    DevArray<double> part;
    DevArray<MState> st;
    MState* h = nullptr;                // pinned, two slots
    hipEvent_t ev[2] = {nullptr, nullptr};
    ~MultiWork()
    {
        if (h) (void)hipHostFree(h);
        for (hipEvent_t e : ev)
            if (e) (void)hipEventDestroy(e);
    }
};

// Grid of a row-tile kernel: as many workgroups as are resident at once (occupancy per CU times the
// CUs), at most kMGrid and one per tile. Each workgroup takes a contiguous range of tiles, so with the whole grid
// resident from the start no workgroup waits for a second round.
template <typename K>
static int resident_grid(K kernel, int ntiles)
{
    int per_cu = 0, dev = 0, cus = 0;
    PFEM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, reinterpret_cast<const void*>(kernel), kMBlock, 0));
    PFEM_HIP(hipGetDevice(&dev));
    PFEM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev));
    const int most = std::max(8, std::min(kMGrid, per_cu * cus) / 8 * 8);
    return std::min(most, (ntiles + 7) / 8 * 8);
}

// Polls the state every `batch` iterations until every column is done (or `slots` are spent), one batch ahead
// of the copy it waits for. iterate() launches one iteration.
template <typename F>
static void m_iterate(Context* c, MultiWork& w, int batch, int slots, F iterate)
{
    int launched = 0, pend = -1, slot = 0;
    while (true) {
        for (int jb = 0; jb < batch; ++jb) iterate();
        launched += batch;
        PFEM_HIP(hipGetLastError());
        PFEM_HIP(hipMemcpyAsync(w.h + slot, w.st.p, sizeof(MState), hipMemcpyDeviceToHost, c->stream));
        PFEM_HIP(hipEventRecord(w.ev[slot], c->stream));
        if (pend >= 0) {
            PFEM_HIP(hipEventSynchronize(w.ev[pend]));
            if (w.h[pend].all_done || launched > slots + 2 * batch) break;
        }
        pend = slot;
        slot ^= 1;
    }
}

static void m_state(Context* c, pfem_solver_t* s, MultiWork& w)
{
    MState init[2]{};
    init[0].tol = s->tol;
    init[0].tol_mode = s->tol_mode;
    init[0].maxit = s->maxit;
    init[0].ncol = w.ncol;
    init[0].drop = std::pow(10.0, -s->replace_digits);
    init[1] = init[0];
    PFEM_HIP(hipMemcpyAsync(w.st.p, init, sizeof init, hipMemcpyHostToDevice, c->stream));
}

// FP64 CG over the interleaved system. Ends with the state in h[0].
template <int G, bool JAC>
static void m_cg_run(Context* c, pfem_solver_t* s, MultiWork& w, const Pattern& P, pfem_csr_t* a)
{
    const int n = P.n;
    const double* invd = JAC ? s->pc->invd.p : nullptr;
    const double* val = a->val.p;
    double *x = w.x.p, *b = w.b.p, *r = w.r.p, *p = w.p.p, *q = w.q.p;
    MState *s0 = w.st.p, *s1 = w.st.p + 1;
    m_state(c, s, w);
    double* pa = w.part.p;
    double* pb = w.part.p + (size_t)2 * G * kMGrid;
    const int ni = resident_grid(k_m_init<G, JAC>, w.ntiles), ns = resident_grid(k_m_spmv<G>, w.ntiles);
    const int nu = (int)std::min<long>(kMStream, ((long)n * G + kMBlock - 1) / kMBlock);
    const dim3 bl(kMBlock);
    hipLaunchKernelGGL((k_m_init<G, JAC>), dim3(ni), bl, 0, c->stream, w.ntiles, w.tiles.p, P.rowptr.p, P.col.p, val, x, b, invd, r, p, pa);
    hipLaunchKernelGGL((k_m_begin<G>), dim3(1), bl, 0, c->stream, s0, (const double*)pa, ni);
    PFEM_HIP(hipGetLastError());
    m_iterate(c, w, s->poll, s->maxit, [&] {
        hipLaunchKernelGGL((k_m_spmv<G>), dim3(ns), bl, 0, c->stream, w.ntiles, w.tiles.p, P.rowptr.p, P.col.p, val, p, q, s0, pa);
        hipLaunchKernelGGL((k_m_update<G, JAC>), dim3(nu), bl, 0, c->stream, n, r, q, invd, s0, s1, (const double*)pa, ns, pb);
        hipLaunchKernelGGL((k_m_p<G, JAC>), dim3(nu), bl, 0, c->stream, n, x, p, r, invd, s1, s0, (const double*)pb, nu);
    });
    PFEM_HIP(hipMemcpyAsync(w.h, w.st.p, sizeof(MState), hipMemcpyDeviceToHost, c->stream));
    PFEM_HIP(hipStreamSynchronize(c->stream));
}

// Reliable-update PCG over the interleaved system (x, b in w.x, w.b); ends with the state in h[0]
template <int G, bool JAC>
static void m_ru_run(Context* c, pfem_solver_t* s, MultiWork& w, const Pattern& P, pfem_csr_t* a)
{
    const int n = P.n;
    const size_t m = (size_t)n * G;
    if (!w.x32.p) {
        w.x32.alloc(m); w.r32.alloc(m); w.p32.alloc(m); w.q32.alloc(m);
    }
    if (!a->val32.p) a->val32.alloc(P.nnz);
    hipLaunchKernelGGL(k_m_to32, dim3(blocks_for(P.nnz)), dim3(kBlock), 0, c->stream, (long)P.nnz, a->val32.p, a->val.p);
    const double* invd = JAC ? s->pc->invd.p : nullptr;
    const float* invd32 = JAC ? s->pc->invd32.p : nullptr;
    PFEM_REQUIRE(!JAC || invd32, "FP32 Jacobi diagonal missing");
    MState *s0 = w.st.p, *s1 = w.st.p + 1;
    m_state(c, s, w);
    double* pa = w.part.p;
    double* pb = w.part.p + (size_t)2 * G * kMGrid;
    float *xs = w.x32.p, *rs = w.r32.p, *ps = w.p32.p, *qs = w.q32.p;
    const int ni = resident_grid(k_mr_init<G, JAC>, w.ntiles), ns = resident_grid(k_mr_spmv<G, JAC>, w.ntiles);
    const int nu = (int)std::min<long>(kMStream, ((long)n * G + kMBlock - 1) / kMBlock);
    const dim3 bl(kMBlock);
    hipLaunchKernelGGL((k_mr_init<G, JAC>), dim3(ni), bl, 0, c->stream, w.ntiles, w.tiles.p, P.rowptr.p, P.col.p, a->val.p, (const double*)w.x.p, (const double*)w.b.p, invd, invd32, rs, ps, xs, pa);
    hipLaunchKernelGGL((k_m_begin<G>), dim3(1), bl, 0, c->stream, s0, (const double*)pa, ni);
    PFEM_HIP(hipGetLastError());
    // a replacement takes one extra slot per tenfold residual drop; the slot budget allows for them
    m_iterate(c, w, s->poll, s->maxit + s->maxit / 4 + 64, [&] {
        hipLaunchKernelGGL((k_mr_spmv<G, JAC>), dim3(ns), bl, 0, c->stream, w.ntiles, w.tiles.p, P.rowptr.p, P.col.p, (const float*)a->val32.p, (const double*)a->val.p, (const float*)ps, qs, (const double*)w.x.p, (const double*)w.b.p, invd, rs, s0, pa);
        hipLaunchKernelGGL((k_mr_update<G, JAC>), dim3(nu), bl, 0, c->stream, n, rs, (const float*)qs, invd32, s0, s1, (const double*)pa, ns, pb);
        hipLaunchKernelGGL((k_mr_p<G, JAC>), dim3(nu), bl, 0, c->stream, n, ps, (const float*)rs, invd32, w.x.p, xs, s1, s0, (const double*)pb, nu);
    });
    // columns still iterating at the slot limit keep their FP64 part; their FP32 correction is folded in
    hipLaunchKernelGGL(k_mr_fold, dim3(blocks_for((long)m)), dim3(kBlock), 0, c->stream, (long)m, w.x.p, (const float*)xs);
    PFEM_HIP(hipMemcpyAsync(w.h, w.st.p, sizeof(MState), hipMemcpyDeviceToHost, c->stream));
    PFEM_HIP(hipStreamSynchronize(c->stream));
}

template <int G>
static void solve_multi_g(Context* c, pfem_solver_t* s, pfem_csr_t* a, int ncol, double* X, const double* B,
                          pfem_solve_stats* stats)
{
    const Pattern& P = *a->pat;
    const int n = P.n;
    if (!s->multi || s->multi->G != G || s->multi->n != n || s->multi->pat != a->pat) {
        s->multi.reset(new MultiWork());
        MultiWork& w = *s->multi;
        w.n = n;
        w.G = G;
        w.pat = a->pat;
        std::vector<int> tiles;
        for (int r = 0; r < n;) {
            int r1 = r;
            const int base = P.h_rowptr[r];
            while (r1 < n && r1 - r < tile_rows<G> && (P.h_rowptr[r1 + 1] - base <= kMTileNnz || r1 == r)) ++r1;
            tiles.push_back(r);
            tiles.push_back(r1);
            r = r1;
        }
        w.ntiles = (int)tiles.size() / 2;
        upload(c, w.tiles, tiles);
        const size_t m = (size_t)n * G;
        w.x.alloc(m); w.b.alloc(m); w.r.alloc(m); w.p.alloc(m); w.q.alloc(m);
        w.part.alloc((size_t)4 * G * kMGrid);
        w.st.alloc(2);
        PFEM_HIP(hipHostMalloc((void**)&w.h, 2 * sizeof(MState), hipHostMallocDefault));
        for (hipEvent_t& e : w.ev) PFEM_HIP(hipEventCreateWithFlags(&e, hipEventDisableTiming));
    }
    MultiWork& w = *s->multi;
    w.ncol = ncol;
    const size_t m = (size_t)n * G;
    const unsigned gp = (unsigned)std::min<size_t>(blocks_for((long)m), 8192);
    const bool jac = s->pc && s->pc->kind == PFEM_PRECOND_JACOBI;
    if (s->pc) precond_initialize(c, s->pc, a);
    hipLaunchKernelGGL((k_m_pack<G, double>), dim3(gp), dim3(kBlock), 0, c->stream, n, ncol, (const double*)X, w.x.p);
    hipLaunchKernelGGL((k_m_pack<G, double>), dim3(gp), dim3(kBlock), 0, c->stream, n, ncol, B, w.b.p);
    std::vector<pfem_solve_stats> st(ncol);
    const bool mixed = s->precision == PFEM_PRECISION_MIXED;
    if (mixed && jac) m_ru_run<G, true>(c, s, w, P, a);
    else if (mixed) m_ru_run<G, false>(c, s, w, P, a);
    else if (jac) m_cg_run<G, true>(c, s, w, P, a);
    else m_cg_run<G, false>(c, s, w, P, a);
    for (int j = 0; j < ncol; ++j) {
        const MCol& e = w.h->col[j];
        st[j].converged = e.converged;
        st[j].iterations = e.it;
        st[j].final_residual = e.res;
        st[j].nan_detected = e.nan;
        if (mixed) st[j].refinements = e.nrep;
    }
    hipLaunchKernelGGL((k_m_unpack<G>), dim3(gp), dim3(kBlock), 0, c->stream, n, ncol, (const double*)w.x.p, X);
    PFEM_HIP(hipGetLastError());
    PFEM_HIP(hipStreamSynchronize(c->stream));
    if (stats) std::memcpy(stats, st.data(), sizeof(pfem_solve_stats) * ncol);
}

void MultiWorkDeleter::operator()(MultiWork* w) const { delete w; }

}  // namespace pfem

using namespace pfem;

extern "C" {

int pfem_solver_solve_multi(pfem_solver s, pfem_csr a, int nrhs, double* d_X, const double* d_B,
                            pfem_solve_stats* stats)
{
    PFEM_TRY(s ? s->ctx : nullptr, {
        PFEM_REQUIRE(s && a && d_X && d_B, "null argument");
        PFEM_REQUIRE(nrhs >= 1 && nrhs <= kMaxRhs, "nrhs must be 1..8");
        PFEM_REQUIRE(a->pat->n == s->n, "matrix size differs from the solver's");
        PFEM_REQUIRE(s->kind == PFEM_SOLVER_CG, "multi-RHS solves are PCG only");
        PFEM_REQUIRE(!s->pc || s->pc->kind == PFEM_PRECOND_JACOBI || s->pc->kind == PFEM_PRECOND_NONE,
                     "multi-RHS PCG takes a Jacobi preconditioner or none");
        PFEM_REQUIRE(s->precision == PFEM_PRECISION_FP64 || s->precision == PFEM_PRECISION_MIXED,
                     "multi-RHS PCG runs in FP64 or MIXED precision");
        Context* c = C(s->ctx);
        if (nrhs == 1) solve_multi_g<1>(c, s, a, nrhs, d_X, d_B, stats);
        else if (nrhs == 2) solve_multi_g<2>(c, s, a, nrhs, d_X, d_B, stats);
        else if (nrhs <= 4) solve_multi_g<4>(c, s, a, nrhs, d_X, d_B, stats);
        else solve_multi_g<8>(c, s, a, nrhs, d_X, d_B, stats);
    });
}

}  // extern "C"
