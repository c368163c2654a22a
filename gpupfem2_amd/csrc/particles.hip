// ParticleHandler2D on gfx950 (src/particles/particle_handler_2d.cu).
//
// Layout: structure of arrays (cell, lambda_1..2 as one 16-byte load, lambda_3, position, velocity, ID),
// double buffered for the reorder. The reference's 96-byte AoS record is dragged through every kernel;
// here each kernel touches only the fields it needs.
//
// Per step (advect): one kernel advects and relocates every particle through all substeps (the
// substeps only depend on the particle itself and the fixed velocity field) and takes the census: per cell
// an occupied-subcell mask and the live particles; a particle outside its cell's 1-ring is marked dead. A
// prefix sum over the cells gives every cell its places in the other buffer, empty subcells are refilled
// there (IDs in (cell, subcell) order), and the particles are copied to their places, stably by cell (dead
// particles dropped). The sorted order is what makes the projection a deterministic segmented reduction:
// per cell over its contiguous particle range, then per node over its incident cells -- no atomics (the
// reference uses 9 FP64 atomicAdd per particle, :90-107).
//
// The particle count lives on the device ({count, next ID, deleted, added} in pst): every kernel of a step
// reads it there and is launched over the buffers' capacity, which the host keeps at least the count plus
// the largest possible refill (one particle per subcell of every cell), so a step never waits for the
// device to report how many particles it added or deleted. The host learns the new count from an
// asynchronous copy read at its next use (the next step's capacity check, pfem_particles_count); by then
// the stream has long passed it. With fixed capacity and no host-side count, a step's particle kernels
// are the same launch sequence every step (two sequences: the buffers alternate), which the stepper can
// replay from a HIP graph.
#include <algorithm>
#include <cmath>
#include <cstring>

#include "device.hpp"
#include "internal.hpp"

struct pfem_particles_t {
    pfem_ctx ctx = nullptr;
    pfem_mesh2d_t* mesh = nullptr;
    int level = 2, ns = 4;
    double centers[16][3];
    long count = 0, capacity = 0;
    uint32_t next_id = 0;
    int cur = 0;
    pfem::DevArray<int> cell[2];
    pfem::DevArray<double2> lam12[2];
    pfem::DevArray<double> lam3[2];
    pfem::DevArray<double2> pos[2], vel[2];
    pfem::DevArray<uint32_t> id[2];
    // per cell: occupied subcells, live particles, the refill's and the cells' prefix sums, the next free place
    // (live and counters {deleted, -, long cells, cells of k_proj_crowded} lie behind mask; those cells' list has the
    // place of the cells' next free places, which only the reorder uses)
    pfem::DevArray<uint32_t> mask;
    int *live = nullptr, *counters = nullptr;
    pfem::DevArray<int> cursor, cell_start;
    pfem::DevArray<unsigned long long> prefix, tile_sums;
    // the particle that goes to each place, in any order within a cell; the first cell of each reorder tile;
    // cells with more particles than a workgroup orders in LDS
    pfem::DevArray<uint32_t> order, order2;
    pfem::DevArray<int> tile_cell, long_cells, left_n;
    pfem::DevArray<double> part;
    long deleted_last = 0, added_last = 0;
    // device state {count, next ID, deleted, added} of the last step, its pinned host copy and the event
    // that completes the copy; generation counts reallocations of the particle buffers
    pfem::DevArray<long> pst;
    long* h_pst = nullptr;
    hipEvent_t pst_ev = nullptr;
    bool pst_pending = false;
    long generation = 0;
    ~pfem_particles_t()
    {
        if (pst_ev) (void)hipEventDestroy(pst_ev);
        if (h_pst) (void)hipHostFree(h_pst);
    }
};

namespace pfem {

struct Centers {
    double c[16][3];
};

// ------------------------------------------------------------------ Philox4x32-10
// Salmon, Moraes, Dror, Shaw, "Parallel random numbers: as easy as 1, 2, 3" (SC'11)
__device__ __forceinline__ uint4 philox4x32_10(uint4 c, uint2 k)
{
#pragma unroll
    for (int r = 0; r < 10; ++r) {
        const uint32_t hi0 = __umulhi(0xD2511F53u, c.x), lo0 = 0xD2511F53u * c.x;
        const uint32_t hi1 = __umulhi(0xCD9E8D57u, c.z), lo1 = 0xCD9E8D57u * c.z;
        c = make_uint4(hi1 ^ c.y ^ k.x, lo1, hi0 ^ c.w ^ k.y, lo0);
        k.x += 0x9E3779B9u;
        k.y += 0xBB67AE85u;
    }
    return c;
}

__device__ __forceinline__ double u01(uint32_t a, uint32_t b)
{
    return ((double)(a >> 5) * 67108864.0 + (double)(b >> 6)) * (1.0 / 9007199254740992.0);
}

// determineSubcell (particle_handler_2d.cu:10-33), row/column clamped to the triangle (the reference
// indexes past the cell's counters for particles inside the 2e-6 tolerance band below/right of it)
__device__ __forceinline__ int subcell(int L, double step, double l1, double l2, double l3)
{
    int i = (int)((1.0 - l2) * L);
    i = i > L - 1 ? L - 1 : (i < 0 ? 0 : i);
    int j = (int)(l1 * L);
    j = j > i ? i : (j < 0 ? 0 : j);
    int res = i * i + 2 * j;
    if (j != i) {
        const double x = step * (j + 1);
        const double y = 1.0 - step * (i + 1);
        const double z = 1.0 - x - y;
        if (l3 < z) ++res;
    }
    return res;
}

// ------------------------------------------------------------------ kernels
// kSeedParticlesIntoCell (particle_handler_2d.cu:35-52), deterministic: particle k of cell c at c*ppc + k
__global__ void k_seed(int nt, int ppc, int mode, const double* __restrict__ xy, const int* __restrict__ tri,
                       Centers cen, uint2 key, int* __restrict__ cell, double2* __restrict__ lam12,
                       double* __restrict__ lam3, double2* __restrict__ pos, double2* __restrict__ vel,
                       uint32_t* __restrict__ id)
{
    const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= (long)nt * ppc) return;
    const int c = (int)(p / ppc), k = (int)(p % ppc);
    double L0, L1, L2;
    if (mode == 0) {
        L0 = cen.c[k][0]; L1 = cen.c[k][1]; L2 = cen.c[k][2];
    } else {
        const uint4 r = philox4x32_10(make_uint4((uint32_t)c, (uint32_t)k, 0u, 0u), key);
        const double s = sqrt(u01(r.x, r.y));
        const double r2 = u01(r.z, r.w);
        L0 = 1.0 - s; L1 = s * (1.0 - r2); L2 = s * r2;
    }
    const int a = tri[3 * c], b = tri[3 * c + 1], d = tri[3 * c + 2];
    cell[p] = c;
    lam12[p] = make_double2(L0, L1);
    lam3[p] = L2;
    pos[p] = make_double2(L0 * xy[2 * a] + L1 * xy[2 * b] + L2 * xy[2 * d],
                          L0 * xy[2 * a + 1] + L1 * xy[2 * b + 1] + L2 * xy[2 * d + 1]);
    vel[p] = make_double2(0.0, 0.0);
    id[p] = (uint32_t)p;
}

// kCorrectParticleVelocity (particle_handler_2d.cu:72-88); uo == nullptr is initParticleVelocity
__global__ void k_correct(const long* __restrict__ pst, const int* __restrict__ cell, const double2* __restrict__ lam12,
                          const double* __restrict__ lam3, double2* __restrict__ vel, const int* __restrict__ tri,
                          const double* __restrict__ u0, const double* __restrict__ u1,
                          const double* __restrict__ uo0, const double* __restrict__ uo1)
{
    const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (p >= pst[0]) return;
    const int c = cell[p];
    const double2 l12 = lam12[p];
    const double l[3] = {l12.x, l12.y, lam3[p]};
    double ix = 0.0, iy = 0.0;
    for (int i = 0; i < 3; ++i) {
        const int v = tri[3 * c + i];
        ix += l[i] * (u0[v] - (uo0 ? uo0[v] : 0.0));
        iy += l[i] * (u1[v] - (uo1 ? uo1[v] : 0.0));
    }
    double2 vv = vel[p];
    vv.x = vv.x + ix;
    vv.y = vv.y + iy;
    vel[p] = vv;
}

// Particle2D::isInsideCell (particle_2d.cu:14-22), GEOMETRY::transformGlobalToLocal and
// isPointInsideUnitTriangle (geometry.cuh:14-46)
__device__ __forceinline__ bool inside(const double4 J, double v3x, double v3y, double px, double py, double* L)
{
    const double dx = px - v3x, dy = py - v3y;
    L[0] = J.x * dx + J.z * dy;
    L[1] = J.y * dx + J.w * dy;
    L[2] = 1.0 - L[0] - L[1];
#pragma unroll
    for (int d = 0; d < 3; ++d)
        if (L[d] > 1.0 + 2e-6 || L[d] < -2e-6) return false;
    return true;
}

// Runs of equal cells over the wave's lanes (cell -1: none): whether this lane begins one, and its length
// there. Particles arrive grouped by cell and advection moves few of them, so a wave holds a few runs and
// one atomic per run and counter replaces one per particle.
__device__ __forceinline__ bool cell_run(int c, int lane, int& length)
{
    const int prev = __shfl_up(c, 1, 64);
    const bool head = lane == 0 || prev != c;
    const unsigned long long heads = __ballot(head);
    const unsigned long long after = lane < 63 ? heads >> (lane + 1) : 0ull;
    length = after ? __ffsll((unsigned long long)after) : 64 - lane;
    return head;
}

// All substeps of advectParticles (particle_handler_2d.cu:328-338): kAdvectParticles (:54-70) then the
// relocation of sortParticlesInCells (:363-395): own cell, then the vertex neighbours ascending, first
// hit wins; a particle found nowhere is marked dead (cell = -1). Then the census of
// kCountParticlesInSubcells (:173-181): the subcell bits (only emptiness matters) and the live particles of
// every cell.
//
// Two launches. The first advances every particle until it leaves its cell: 44 bytes read and written a
// particle, its cell's geometry and nodal velocities loaded once for all substeps. The few that leave (1 to
// 5% a substep) are listed per workgroup, and the second launch searches for them and advances them to the
// end, with full waves of such particles: a search is a chain of a dozen candidates, and one leaving particle
// made its whole wave wait for it (in one launch, even with 16 lanes testing one particle's candidates at
// once: 1.71 ms for 53M particles and 146 us for 3M; here 0.92 + 0.45 ms and 64 + 78 us).
struct CellField {   // a cell's geometry and nodal velocities
    double4 J;
    double2 o;
    double a0, a1, a2, b0, b1, b2;
};

__device__ __forceinline__ void load_cell(CellField& f, int c, const int* __restrict__ tri, const double4* __restrict__ invJ,
                                          const double2* __restrict__ v3, const double* __restrict__ u0,
                                          const double* __restrict__ u1)
{
    const int t0 = tri[3 * c], t1 = tri[3 * c + 1], t2 = tri[3 * c + 2];
    f.J = invJ[c];
    f.o = v3[c];
    f.a0 = u0[t0]; f.a1 = u0[t1]; f.a2 = u0[t2];
    f.b0 = u1[t0]; f.b1 = u1[t1]; f.b2 = u1[t2];
}

// One substep: x moves; l follows while x stays in the cell (false: it left)
__device__ __forceinline__ bool substep(const CellField& f, double dts, double2& x, double (&l)[3])
{
    double ax = 0.0, ay = 0.0;
    ax += l[0] * f.a0; ay += l[0] * f.b0;
    ax += l[1] * f.a1; ay += l[1] * f.b1;
    ax += l[2] * f.a2; ay += l[2] * f.b2;
    x.x = x.x + dts * ax;
    x.y = x.y + dts * ay;
    double M[3];
    if (!inside(f.J, f.o.x, f.o.y, x.x, x.y, M)) return false;
    l[0] = M[0]; l[1] = M[1]; l[2] = M[2];
    return true;
}

// The one cell of a wave's particles (c = -1: none), -1 if there are none, -2 if there are several; of one cell
// also the particles' number and subcells
__device__ __forceinline__ int one_cell(int c, uint32_t& bits, int& number)
{
    const unsigned long long here = __ballot(c >= 0);
    if (!here) return -1;
    const int one = __builtin_amdgcn_readlane(c, __ffsll(here) - 1);
    if (!__all(c < 0 || c == one)) return -2;
    number = __popcll(here);
    if (c < 0) bits = 0u;
#pragma unroll
    for (int off = 32; off > 0; off >>= 1) bits |= __shfl_xor(bits, off, 64);
    return one;
}

// The census of a wave's particles (c = -1: none)
__device__ __forceinline__ void census(int c, uint32_t bits, int lane, uint32_t* __restrict__ mask, int* __restrict__ live)
{
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const uint32_t ob = __shfl_down(bits, off, 64);
        const int oc = __shfl_down(c, off, 64);
        if (lane + off < 64 && oc == c) bits |= ob;
    }
    int length;
    if (cell_run(c, lane, length) && c >= 0) {
        atomicOr(&mask[c], bits);
        atomicAdd(&live[c], length);
    }
}

// Particles that leave their cell in substep s: {particle, s} into left_p / left_s, a range of kBlock per
// workgroup, their number in left_n. A workgroup whose particles share one cell takes its census at once: the atomics
// of a crowded cell all meet in one place (1M particles in one cell: 1.91 -> 0.18 ms).
__global__ __launch_bounds__(kBlock) void k_advect(
    const long* __restrict__ pst, int substeps, double dts, const int* __restrict__ cell, double2* __restrict__ lam12,
    double* __restrict__ lam3, double2* __restrict__ pos, const int* __restrict__ tri, const double4* __restrict__ invJ,
    const double2* __restrict__ v3, const double* __restrict__ u0, const double* __restrict__ u1, int L, double step,
    uint32_t* __restrict__ mask, int* __restrict__ live, uint32_t* __restrict__ left_p, uint32_t* __restrict__ left_s,
    int* __restrict__ left_n)
{
    __shared__ int wn[kWaves], wc[kWaves], wl[kWaves];
    __shared__ uint32_t wb[kWaves];
    const long p = (long)blockIdx.x * kBlock + threadIdx.x;
    const long P = pst[0];
    if ((long)blockIdx.x * kBlock >= P) return;   // a whole workgroup past the count (the grid covers the capacity)
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int c = -1, s = 0;
    uint32_t bits = 0u;
    bool leaves = false;
    if (p < P) {
        c = cell[p];
        const double2 l12 = lam12[p];
        double l[3] = {l12.x, l12.y, lam3[p]};
        double2 x = pos[p];
        CellField f;
        load_cell(f, c, tri, invJ, v3, u0, u1);
        for (; s < substeps && !leaves; ++s) leaves = !substep(f, dts, x, l);
        lam12[p] = make_double2(l[0], l[1]);
        lam3[p] = l[2];
        pos[p] = x;
        bits = 1u << subcell(L, step, l[0], l[1], l[2]);
    }
    const unsigned long long left = __ballot(leaves);
    const int stays = leaves ? -1 : c;
    uint32_t subcells = bits;
    int number = 0;
    const int one = one_cell(stays, subcells, number);
    if (lane == 0) {
        wn[wid] = __popcll(left);
        wc[wid] = one;
        wl[wid] = number;
        wb[wid] = subcells;
    }
    __syncthreads();
    int at = 0, all = 0, shared = -1;
    number = 0;
    subcells = 0u;
    for (int w = 0; w < kWaves; ++w) {
        if (w < wid) at += wn[w];
        all += wn[w];
        if (wc[w] == -1) continue;
        shared = shared == -1 || shared == wc[w] ? wc[w] : -2;
        number += wl[w];
        subcells |= wb[w];
    }
    if (threadIdx.x == 0) left_n[blockIdx.x] = all;
    if (leaves) {
        const size_t q = (size_t)blockIdx.x * kBlock + at + __popcll(left & ((1ull << lane) - 1ull));
        left_p[q] = (uint32_t)p;
        left_s[q] = (uint32_t)s;   // the substeps taken
    }
    if (shared == -2) {
        census(stays, bits, lane, mask, live);
    } else if (threadIdx.x == 0 && shared >= 0) {
        atomicOr(&mask[shared], subcells);
        atomicAdd(&live[shared], number);
    }
}

// One wave per RANGES lists of k_advect: four make full waves where few particles leave, one gives a set of
// a few million enough waves for the chip. SPLIT waves to a list: a small set, whose waves do not fill the chip, would
// otherwise take a list in which all particles leave 64 at a time (12.8k particles, 20 substeps of half a cell:
// 262 -> 130 us a step, where one kernel with a particle a lane took 208).
template <int RANGES, int SPLIT>
__global__ __launch_bounds__(kBlock) void k_relocate(
    const long* __restrict__ pst, int substeps, double dts, int* __restrict__ cell, double2* __restrict__ lam12,
    double* __restrict__ lam3, double2* __restrict__ pos, const int* __restrict__ tri, const double4* __restrict__ invJ,
    const double2* __restrict__ v3, const int* __restrict__ nbr_off, const int* __restrict__ nbr_idx,
    const double* __restrict__ u0, const double* __restrict__ u1, int L, double step, uint32_t* __restrict__ mask,
    int* __restrict__ live, const uint32_t* __restrict__ left_p, const uint32_t* __restrict__ left_s,
    const int* __restrict__ left_n, int* __restrict__ dead)
{
    const int lane = threadIdx.x & 63;
    const long wave = (long)blockIdx.x * kWaves + (threadIdx.x >> 6), range = wave / SPLIT * RANGES;
    const long ranges = (pst[0] + kBlock - 1) / kBlock;
    if (range >= ranges) return;
    int end[RANGES], total = 0;
#pragma unroll
    for (int r = 0; r < RANGES; ++r) {
        total += range + r < ranges ? left_n[range + r] : 0;
        end[r] = total;
    }
    for (int t0 = 64 * (int)(wave % SPLIT); t0 < total; t0 += 64 * SPLIT) {
        const int t = t0 + lane;
        int c = -1;
        uint32_t bits = 0u;
        bool lost = false;
        if (t < total) {
            int r = 0, before = 0;
#pragma unroll
            for (int k = 0; k < RANGES - 1; ++k)
                if (t >= end[k]) {
                    r = k + 1;
                    before = end[k];
                }
            const size_t q = (size_t)(range + r) * kBlock + (t - before);
            const uint32_t p = left_p[q];
            int s = (int)left_s[q];
            c = cell[p];
            const double2 l12 = lam12[p];
            double l[3] = {l12.x, l12.y, lam3[p]};
            double2 x = pos[p];
            while (true) {
                // x has just left cell c: the candidates in ascending order, four loaded together
                int found = -1;
                double M[3] = {0.0, 0.0, 0.0};
                const int k1 = nbr_off[c + 1];
                for (int k = nbr_off[c]; k < k1 && found < 0; k += 4) {
                    int nb[4];
                    double4 Jn[4];
                    double2 on[4];
#pragma unroll
                    for (int u = 0; u < 4; ++u) nb[u] = nbr_idx[min(k + u, k1 - 1)];
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        Jn[u] = invJ[nb[u]];
                        on[u] = v3[nb[u]];
                    }
#pragma unroll
                    for (int u = 0; u < 4; ++u) {
                        double N[3];
                        if (found < 0 && inside(Jn[u], on[u].x, on[u].y, x.x, x.y, N)) {
                            found = nb[u];   // (a repeated last candidate fails like the first time)
                            M[0] = N[0]; M[1] = N[1]; M[2] = N[2];
                        }
                    }
                }
                c = found;
                if (found < 0) {
                    lost = true;
                    break;
                }
                l[0] = M[0]; l[1] = M[1]; l[2] = M[2];
                bool leaves = false;
                if (s < substeps) {
                    CellField f;
                    load_cell(f, c, tri, invJ, v3, u0, u1);
                    for (; s < substeps && !leaves; ++s) leaves = !substep(f, dts, x, l);
                }
                if (!leaves) break;
            }
            cell[p] = c;
            lam12[p] = make_double2(l[0], l[1]);
            lam3[p] = l[2];
            pos[p] = x;
            if (c >= 0) bits = 1u << subcell(L, step, l[0], l[1], l[2]);
        }
        const unsigned long long gone = __ballot(lost);
        if (gone && lane == 0) atomicAdd(dead, __popcll(gone));
        census(c, bits, lane, mask, live);
    }
}

// ------------------------------------------------------------------ exclusive scan (int)
constexpr int kScanItems = 16;
constexpr int kScanTile = kBlock * kScanItems;

__device__ int block_exclusive_scan(int v, int* total)
{
    __shared__ int wsum[kWaves];
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6;
    int x = v;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
        const int y = __shfl_up(x, off, 64);
        if (lane >= off) x += y;
    }
    if (lane == 63) wsum[wid] = x;
    __syncthreads();
    int pre = 0, tot = 0;
    for (int w = 0; w < kWaves; ++w) {
        if (w < wid) pre += wsum[w];
        tot += wsum[w];
    }
    __syncthreads();
    *total = tot;
    return pre + x - v;
}

__global__ void k_scan_tiles(const int* __restrict__ in, int* __restrict__ out, long n, int* __restrict__ sums)
{
    __shared__ int buf[kScanTile];
    const long base = (long)blockIdx.x * kScanTile;
    for (int i = threadIdx.x; i < kScanTile; i += kBlock) buf[i] = base + i < n ? in[base + i] : 0;
    __syncthreads();
    int run = 0;
    for (int i = 0; i < kScanItems; ++i) run += buf[threadIdx.x * kScanItems + i];
    int tot;
    int pre = block_exclusive_scan(run, &tot);
    for (int i = 0; i < kScanItems; ++i) {
        const int v = buf[threadIdx.x * kScanItems + i];
        buf[threadIdx.x * kScanItems + i] = pre;
        pre += v;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kScanTile; i += kBlock)
        if (base + i < n) out[base + i] = buf[i];
    if (threadIdx.x == 0 && sums) sums[blockIdx.x] = tot;
}

__global__ void k_scan_add(int* __restrict__ out, long n, const int* __restrict__ sums_scanned)
{
    const long base = (long)blockIdx.x * kScanTile;
    const int add = sums_scanned[blockIdx.x];
    for (int i = threadIdx.x; i < kScanTile; i += kBlock)
        if (base + i < n) out[base + i] += add;
}

// total = sum(in) written to total_dev (if not null); tmp holds at least ntiles + ntiles2 + 1 ints
static void scan_with_tmp(Context* c, const int* in, int* out, long n, int* tmp, int* total_dev);

__global__ void k_scan_total(const int* __restrict__ in, const int* __restrict__ out, long n, int* __restrict__ total)
{
    if (threadIdx.x == 0 && blockIdx.x == 0) *total = n > 0 ? out[n - 1] + in[n - 1] : 0;
}

static void scan_with_tmp(Context* c, const int* in, int* out, long n, int* tmp, int* total_dev)
{
    if (n <= 0) return;
    const long nt = (n + kScanTile - 1) / kScanTile;
    if (nt == 1) {
        hipLaunchKernelGGL(k_scan_tiles, dim3(1), dim3(kBlock), 0, c->stream, in, out, n, (int*)nullptr);
    } else {
        int* sums = tmp;
        int* sums_scan = tmp + nt;
        hipLaunchKernelGGL(k_scan_tiles, dim3(nt), dim3(kBlock), 0, c->stream, in, out, n, sums);
        PFEM_REQUIRE(nt <= kScanTile * (long)kScanTile, "scan too long");
        scan_with_tmp(c, sums, sums_scan, nt, tmp + 2 * nt, nullptr);
        hipLaunchKernelGGL(k_scan_add, dim3(nt), dim3(kBlock), 0, c->stream, out, n, sums_scan);
    }
    if (total_dev) hipLaunchKernelGGL(k_scan_total, dim3(1), dim3(64), 0, c->stream, in, out, n, total_dev);
}

static long scan_tmp_size(long n)
{
    long s = 0;
    while (n > kScanTile) {
        n = (n + kScanTile - 1) / kScanTile;
        s += 2 * n;
    }
    return s + 1;
}

void exclusive_scan_int(Context* c, const int* in, int* out, long n, int* total_dev)
{
    DevArray<int> tmp(scan_tmp_size(n));
    scan_with_tmp(c, in, out, n, tmp.p, total_dev);
    PFEM_HIP(hipStreamSynchronize(c->stream));
}

// ------------------------------------------------------------------ reorder by cell
// The particles are already grouped by cell but for the few that moved, so a sort of all of them is not
// needed: the census counts every cell's particles, a prefix sum over the cells gives the places, each
// particle takes a place of its cell (in any order), and a particle's final place follows from its rank
// among its cell's particles, which keeps their order stable and the result deterministic. Refilled
// particles are written straight to their places, the last of their cell.
constexpr int kTileOut = 1024;    // places a workgroup of k_reorder fills
// More particles in a cell are ordered by k_order_long; ranking them is quadratic. A step of 2M particles, ranked and
// ordered: 256 a cell 238 and 315 us, 400 a cell 276 and 332, 512 a cell 315 and 288, 1000 a cell 666 and 292.
constexpr int kLongCell = 512;
constexpr int kWindow = kTileOut + 2 * (kLongCell + 16);

// 64-bit sums {places of a cell: low, refilled: high}: the tile-local exclusive prefixes and the tile sums
__global__ __launch_bounds__(kBlock) void k_cell_tiles(int nt, int ns, const uint32_t* __restrict__ mask,
                                                       const int* __restrict__ live,
                                                       unsigned long long* __restrict__ prefix,
                                                       unsigned long long* __restrict__ sums)
{
    __shared__ int lo[kScanTile], hi[kScanTile];
    const uint32_t full = ns >= 32 ? 0xffffffffu : ((1u << ns) - 1u);
    const int base = blockIdx.x * kScanTile;
    for (int i = threadIdx.x; i < kScanTile; i += kBlock) {
        int add = 0, n = 0;
        if (base + i < nt) {
            add = ns - __popc(mask[base + i] & full);   // kCountParticlesToBeAdded (:183-195)
            n = live[base + i] + add;
        }
        lo[i] = n;
        hi[i] = add;
    }
    __syncthreads();
    int rl = 0, rh = 0;
    for (int i = 0; i < kScanItems; ++i) {
        rl += lo[threadIdx.x * kScanItems + i];
        rh += hi[threadIdx.x * kScanItems + i];
    }
    int tl, th;
    int pl = block_exclusive_scan(rl, &tl), ph = block_exclusive_scan(rh, &th);
    for (int i = 0; i < kScanItems; ++i) {
        const int k = threadIdx.x * kScanItems + i, vl = lo[k], vh = hi[k];
        lo[k] = pl;
        hi[k] = ph;
        pl += vl;
        ph += vh;
    }
    __syncthreads();
    for (int i = threadIdx.x; i < kScanTile; i += kBlock)
        if (base + i < nt) prefix[base + i] = ((unsigned long long)(unsigned)hi[i] << 32) | (unsigned)lo[i];
    if (threadIdx.x == 0) sums[blockIdx.x] = ((unsigned long long)(unsigned)th << 32) | (unsigned)tl;
}

// Exclusive prefixes of the tile sums, in place, by one workgroup; the step's new state to pst[4..7]: the
// count, the next free ID, the deleted and the added particles (pst[0..3] stay the old ones until the
// reorder's end). Neither 32-bit half overflows: the places are at most the capacity.
__global__ __launch_bounds__(kBlock) void k_cell_top(int ntiles, unsigned long long* __restrict__ sums,
                                                     const int* __restrict__ counters, long* __restrict__ pst)
{
    unsigned long long run = 0;
    for (int b = 0; b < ntiles; b += kBlock) {
        const int i = b + (int)threadIdx.x;
        const unsigned long long v = i < ntiles ? sums[i] : 0ull;
        int tl, th;
        const int pl = block_exclusive_scan((int)(unsigned)v, &tl), ph = block_exclusive_scan((int)(v >> 32), &th);
        if (i < ntiles) sums[i] = run + (((unsigned long long)(unsigned)ph << 32) | (unsigned)pl);
        run += ((unsigned long long)(unsigned)th << 32) | (unsigned)tl;
    }
    if (threadIdx.x == 0) {
        const long added = (long)(run >> 32);
        pst[4] = (long)(unsigned)run;
        pst[5] = pst[1] + added;
        pst[6] = counters[0];
        pst[7] = added;
    }
}

// Per cell: its places [start[c], start[c + 1]); the last ones are the refill's, marked with the cell
constexpr uint32_t kRefill = 0x80000000u;

__global__ void k_cells(int nt, const long* __restrict__ pst, const int* __restrict__ live,
                        const unsigned long long* __restrict__ prefix, const unsigned long long* __restrict__ sums,
                        const uint32_t* __restrict__ mask, int ns, int* __restrict__ start, int* __restrict__ cursor,
                        uint32_t* __restrict__ order, int* __restrict__ tile_cell, int* __restrict__ long_cells,
                        int* __restrict__ counters)
{
    const int c = blockIdx.x * blockDim.x + threadIdx.x;
    if (c > nt) return;
    if (c == nt) {
        start[nt] = (int)pst[4];
        return;
    }
    const int first = (int)(unsigned)(prefix[c] + sums[c / kScanTile]), n = live[c];
    const uint32_t full = ns >= 32 ? 0xffffffffu : ((1u << ns) - 1u);
    const int last = first + n + ns - __popc(mask[c] & full);
    start[c] = first;
    cursor[c] = first;
    for (int t = (first + kTileOut - 1) / kTileOut; (long)t * kTileOut < last; ++t) tile_cell[t] = c;
    if (n > kLongCell) long_cells[atomicAdd(&counters[2], 1)] = c;
    for (int p = first + n; p < last; ++p) order[p] = kRefill | (uint32_t)c;
}

// Every live particle takes a place of its cell (in `list`, if k_order_long sorts the cell): the lanes of a run of
// equal cells take theirs together
// (kPlaceRuns waves' worth of particles per wave, so that their atomics overlap: 0.29 -> 0.19 ms for 53M). Of a
// crowded cell's atomics, which all meet in one place, a wave makes one (1M particles in one cell: 1.16 -> 0.95 ms).
constexpr int kPlaceRuns = 4;

__global__ __launch_bounds__(kBlock) void k_place(const long* __restrict__ pst, const int* __restrict__ cell,
                                                  const int* __restrict__ live, int* __restrict__ cursor,
                                                  uint32_t* __restrict__ order, uint32_t* __restrict__ list)
{
    const long P = pst[0];
    const int lane = threadIdx.x & 63;
    const long p0 = ((long)blockIdx.x * kBlock + (threadIdx.x & ~63)) * kPlaceRuns + lane;
    if ((long)blockIdx.x * kBlock * kPlaceRuns >= P) return;
    int c[kPlaceRuns], at[kPlaceRuns], h[kPlaceRuns];
#pragma unroll
    for (int r = 0; r < kPlaceRuns; ++r) c[r] = p0 + 64 * r < P ? cell[p0 + 64 * r] : -1;
    // the cell of the first particle, if half of the wave's particles are in it: one atomic for all of them
    const int first = __builtin_amdgcn_readfirstlane(c[0]);
    unsigned long long in[kPlaceRuns];
    int many = 0;
#pragma unroll
    for (int r = 0; r < kPlaceRuns; ++r) {
        in[r] = __ballot(c[r] == first);
        many += __popcll(in[r]);
    }
    if (first >= 0 && many >= 32 * kPlaceRuns) {
        int base = 0;
        if (lane == 0) base = atomicAdd(&cursor[first], many);
        base = __builtin_amdgcn_readfirstlane(base);
        uint32_t* __restrict__ const to = live[first] > kLongCell ? list : order;
#pragma unroll
        for (int r = 0; r < kPlaceRuns; ++r) {
            if (c[r] == first) {
                to[base + __popcll(in[r] & ((1ull << lane) - 1ull))] = (uint32_t)(p0 + 64 * r);
                c[r] = -1;
            }
            base += __popcll(in[r]);
        }
    }
#pragma unroll
    for (int r = 0; r < kPlaceRuns; ++r) {
        int length;
        const bool head = cell_run(c[r], lane, length);
        const unsigned long long heads = __ballot(head);
        h[r] = 63 - __clzll((long long)(heads & (~0ull >> (63 - lane))));   // this run's first lane
        at[r] = 0;
        if (head && c[r] >= 0) {
            const bool crowded = live[c[r]] > kLongCell;
            at[r] = atomicAdd(&cursor[c[r]], length);
            if (crowded) at[r] = ~at[r];
        }
    }
#pragma unroll
    for (int r = 0; r < kPlaceRuns; ++r) {
        const int a = __shfl(at[r], h[r], 64);
        if (c[r] < 0) continue;
        if (a >= 0) order[a + lane - h[r]] = (uint32_t)(p0 + 64 * r);
        else list[~a + lane - h[r]] = (uint32_t)(p0 + 64 * r);
    }
}

// Cells of more than kLongCell particles: the particles that took their places (in `list`, in any order) into `order`
// in ascending order. The particles' indices are distinct, so one bit each in LDS sorts them: a pass of a
// workgroup marks those of one window of 2^kOrderShift indices, counts the smaller ones and writes the marked ones
// out behind them. A cell's particles come from its own range of the array and its neighbours' ranges, mostly in
// runs of consecutive indices: a run is marked at once, and windows without particles are passed over. Where
// there are fewer such cells than workgroups, a team of workgroups takes a cell's windows in turn. 1M particles in
// one cell: 13.2 -> 0.25 ms, against radix passes by one workgroup.
constexpr int kOrderLanes = 1024, kOrderBlocks = 256, kOrderShift = 17;

__global__ __launch_bounds__(kOrderLanes) void k_order_long(const int* __restrict__ counters,
                                                            const int* __restrict__ long_cells,
                                                            const int* __restrict__ start, const int* __restrict__ live,
                                                            const uint32_t* __restrict__ list, uint32_t* __restrict__ order)
{
    constexpr int kW = kOrderLanes / 64, kWords = (1 << kOrderShift) / 64, kGroups = kWords / kOrderLanes;
    constexpr int kU = 8;
    __shared__ unsigned long long bits[kWords];
    __shared__ uint32_t least;
    __shared__ int below, wn[kW];
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6, nlong = counters[2];
    int teams = 1;
    while (nlong > 0 && 2 * teams * nlong <= kOrderBlocks) teams *= 2;
    const uint32_t turn = blockIdx.x & (teams - 1);
    for (int q = blockIdx.x / teams; q < nlong; q += kOrderBlocks / teams) {
        const int c = long_cells[q], n = live[c], first = start[c];
        const uint32_t* __restrict__ src = list + first;
        auto ours = [&](uint32_t key) { return ((key >> kOrderShift) & (teams - 1)) == turn; };
        auto publish_least = [&](uint32_t m) {
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) m = min(m, (uint32_t)__shfl_down(m, off, 64));
            if (lane == 0) atomicMin(&least, m);
        };
        __syncthreads();
        if (tid == 0) least = ~0u;
        __syncthreads();
        uint32_t m = ~0u;
        for (int i0 = tid; i0 < n; i0 += kU * kOrderLanes)
#pragma unroll
            for (int u = 0; u < kU; ++u) {
                const int i = i0 + u * kOrderLanes;
                const uint32_t key = src[min(i, n - 1)];
                if (ours(key)) m = min(m, key);
            }
        publish_least(m);
        __syncthreads();
        while (least != ~0u) {
            const uint32_t w0 = least >> kOrderShift << kOrderShift;
            __syncthreads();
            if (tid == 0) {
                least = ~0u;
                below = 0;
            }
            for (int w = tid; w < kWords; w += kOrderLanes) bits[w] = 0ull;
            __syncthreads();
            m = ~0u;
            int smaller = 0;
            for (int i0 = 0; i0 < n; i0 += kU * kOrderLanes) {
                uint32_t keys[kU];
#pragma unroll
                for (int u = 0; u < kU; ++u) keys[u] = src[min(i0 + u * kOrderLanes + tid, n - 1)];
#pragma unroll
                for (int u = 0; u < kU; ++u) {
                    const bool valid = i0 + u * kOrderLanes + tid < n;
                    const uint32_t key = keys[u], d = key - w0;
                    const bool in = valid && d < (1u << kOrderShift);
                    if (valid && key < w0) ++smaller;
                    else if (valid && !in && ours(key)) m = min(m, key);
                    // runs of consecutive indices over the wave's lanes: the first lane marks its run
                    const unsigned long long ins = __ballot(in);
                    if (!ins) continue;
                    const uint32_t before = __shfl_up(d, 1, 64);
                    const bool head = in && (lane == 0 || !((ins >> (lane - 1)) & 1ull) || d != before + 1u);
                    const unsigned long long stops = __ballot(head) | ~ins;
                    if (head) {
                        const unsigned long long after = lane < 63 ? stops >> (lane + 1) : 0ull;
                        const int len = after ? __ffsll(after) : 64 - lane, at = (int)(d & 63u);
                        const unsigned long long ones = ~0ull >> (64 - len);
                        atomicOr(&bits[d >> 6], ones << at);
                        if (at + len > 64) atomicOr(&bits[(d >> 6) + 1], ones >> (64 - at));
                    }
                }
            }
            publish_least(m);
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) smaller += __shfl_down(smaller, off, 64);
            if (lane == 0) atomicAdd(&below, smaller);
            __syncthreads();
            // wave w's words: kGroups groups of 64 from 64 kGroups w on
            int mine = 0;
#pragma unroll
            for (int g = 0; g < kGroups; ++g) mine += __popcll(bits[(wid * kGroups + g) * 64 + lane]);
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) mine += __shfl_down(mine, off, 64);
            if (lane == 0) wn[wid] = mine;
            __syncthreads();
            int at = first + below;
            for (int w = 0; w < wid; ++w) at += wn[w];
            for (int g = 0; g < kGroups; ++g) {
                const int b0 = (wid * kGroups + g) * 64;
                for (unsigned long long some = __ballot(bits[b0 + lane] != 0ull); some; some &= some - 1ull) {
                    const int w = b0 + __ffsll(some) - 1;
                    const unsigned long long word = bits[w];
                    if ((word >> lane) & 1ull) order[at + __popcll(word & ((1ull << lane) - 1ull))] = w0 + 64u * w + lane;
                    at += __popcll(word);
                }
            }
        }
    }
}

// The places of one tile: the particles of the cells that reach into it are ranked in LDS (a particle's
// rank is the number of its cell's particles with a smaller index), then every place's particle is
// copied into the other buffer. A refill place gets kAddParticlesToCell's new particle (:197-236): at the
// centroid of its cell's k-th empty subcell, velocity interpolated from the grid, IDs consecutive from the
// next free one in (cell, subcell) order. Reads and writes 60 and 64 bytes a particle; 53M particles:
// 1.7 ms, 4.1 TB/s; with it the reorder takes 2.0 ms, where a radix sort by cell and a gather took 3.6 ms.
__global__ __launch_bounds__(kBlock) void k_reorder(
    long* __restrict__ pst, int ns, const int* __restrict__ start, const int* __restrict__ live,
    const int* __restrict__ tile_cell, const uint32_t* __restrict__ order, const uint32_t* __restrict__ mask,
    const unsigned long long* __restrict__ prefix, const unsigned long long* __restrict__ sums,
    const double* __restrict__ xy, const int* __restrict__ tri, Centers cen, const double* __restrict__ u0,
    const double* __restrict__ u1, const int* __restrict__ cell0, const double2* __restrict__ l120,
    const double* __restrict__ l30, const double2* __restrict__ pos0, const double2* __restrict__ vel0,
    const uint32_t* __restrict__ id0, int* __restrict__ cell1, double2* __restrict__ l121, double* __restrict__ l31,
    double2* __restrict__ pos1, double2* __restrict__ vel1, uint32_t* __restrict__ id1)
{
    __shared__ uint32_t win[kWindow], perm[kTileOut];
    __shared__ int pcell[kTileOut];
    __shared__ double centre[16][3];
    const long total = pst[4];
    const long tile = (long)blockIdx.x * kTileOut;
    if (tile >= total) return;
    const uint32_t next_id = (uint32_t)(pst[5] - pst[7]);
    const int o0 = (int)tile, o1 = (int)min(total, tile + kTileOut);
    const int cf = tile_cell[blockIdx.x];
    const int lo = live[cf] > kLongCell ? o0 : start[cf];
    int hi = o1;
    if (o1 < total) {
        const int cl = tile_cell[blockIdx.x + 1];
        if (start[cl] < o1 && live[cl] <= kLongCell) hi = start[cl + 1];
    }
    if (threadIdx.x < 48) centre[threadIdx.x / 3][threadIdx.x % 3] = cen.c[threadIdx.x / 3][threadIdx.x % 3];
    for (int j = threadIdx.x; j < hi - lo; j += kBlock) win[j] = order[lo + j];
    __syncthreads();
    for (int j = threadIdx.x; j < hi - lo; j += kBlock) {
        const uint32_t p = win[j];
        int at = lo + j, c = (int)(p & ~kRefill);
        if (!(p & kRefill)) {
            c = cell0[p];
            const int n = live[c], s = start[c];
            if (n <= kLongCell) {
                const uint32_t* w = win + (s - lo);
                int rank = 0;
                for (int k = 0; k < n; ++k) rank += w[k] < p;
                at = s + rank;
            }
        }
        if (at >= o0 && at < o1) {
            perm[at - o0] = p;
            pcell[at - o0] = c;
        }
    }
    __syncthreads();
    constexpr int R = kTileOut / kBlock;
    uint32_t s[R], pid[R];
    double2 l12[R], x[R], v[R];
    double l3[R];
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int j = threadIdx.x + r * kBlock;
        s[r] = j < o1 - o0 ? perm[j] : kRefill;
        if (s[r] & kRefill) continue;
        l12[r] = l120[s[r]];
        l3[r] = l30[s[r]];
        x[r] = pos0[s[r]];
        v[r] = vel0[s[r]];
        pid[r] = id0[s[r]];
    }
#pragma unroll
    for (int r = 0; r < R; ++r) {
        const int j = threadIdx.x + r * kBlock, p = o0 + j;
        if (j >= o1 - o0) continue;
        const int c = pcell[j];
        if (s[r] & kRefill) {
            int k = p - start[c] - live[c];
            pid[r] = next_id + (uint32_t)((prefix[c] + sums[c / kScanTile]) >> 32) + (uint32_t)k;
            uint32_t empty = ~mask[c];
            for (; k > 0; --k) empty &= empty - 1;
            const int q = __ffs(empty) - 1;
            const double L0 = centre[q][0], L1 = centre[q][1], L2 = centre[q][2];
            const int a = tri[3 * c], b = tri[3 * c + 1], d = tri[3 * c + 2];
            l12[r] = make_double2(L0, L1);
            l3[r] = L2;
            x[r] = make_double2(L0 * xy[2 * a] + L1 * xy[2 * b] + L2 * xy[2 * d],
                                L0 * xy[2 * a + 1] + L1 * xy[2 * b + 1] + L2 * xy[2 * d + 1]);
            double vx = 0.0, vy = 0.0;
            vx += L0 * u0[a]; vy += L0 * u1[a];
            vx += L1 * u0[b]; vy += L1 * u1[b];
            vx += L2 * u0[d]; vy += L2 * u1[d];
            v[r] = make_double2(vx, vy);
        }
        cell1[p] = c;
        l121[p] = l12[r];
        l31[p] = l3[r];
        pos1[p] = x[r];
        vel1[p] = v[r];
        id1[p] = pid[r];
    }
}

// The step's new device state (k_cell_top's) in place of the old one
__global__ void k_pstate_finish(long* __restrict__ pst)
{
    if (threadIdx.x < 4 && blockIdx.x == 0) pst[threadIdx.x] = pst[4 + threadIdx.x];
}

__global__ void k_zero_u32(long n, uint32_t* __restrict__ d)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) d[i] = 0u;
}

// first particle of every cell in the cell-sorted array (cell_start[nt] = number of particles)
__global__ void k_cell_start(const long* __restrict__ pst, const int* __restrict__ cell, int nt, int* __restrict__ start)
{
    const long p = (long)blockIdx.x * blockDim.x + threadIdx.x;
    const long n = pst[0];
    if (p > n) return;
    const int prev = p == 0 ? -1 : cell[p - 1];
    const int curc = p == n ? nt : cell[p];
    for (int c = prev + 1; c <= curc; ++c) start[c] = (int)p;
}

// ------------------------------------------------------------------ projection
// kProjectParticleVelocityOntoGrid / kFinalizeVelocityProjection (:90-115) as a segmented reduction
// Per cell the sums of l_i u, l_i v and l_i over its particles, in array order. A workgroup takes 64 cells
// and streams their particles (consecutive in the arrays) through LDS in chunks with coalesced loads; wave
// i sums shape function i of the cells on its lanes. A lane per cell that walks its particles in memory
// instead reads 400 bytes away from its neighbours. 53M particles: 1.23 -> 0.47 ms. Cells of more than kProjMany
// particles are listed for k_proj_crowded: a chunk holds few of them, and most lanes would wait (2M particles, 4000
// a cell: 19.2 ms, here 0.09). Half of the cells on either side of the line is the worst there is, so it lies where
// that is no slower than a lane per cell: 2M particles, us with a line at 32, 64 and 128, all streamed, a lane
// per cell: 64 a cell 68, 78, 57, 53, 76; 100 a cell 63, 71, 89, 85, 106; 128 a cell 60, 63, 125, 121, 130;
// 200 a cell 55, 55, 65, 260, 192.
constexpr int kProjCells = 64, kProjChunk = 1024, kProjMany = 128;

__global__ __launch_bounds__(kBlock) void k_proj_cells(int nt, const int* __restrict__ start,
                                                       const double2* __restrict__ lam12,
                                                       const double* __restrict__ lam3, const double2* __restrict__ vel,
                                                       double* __restrict__ part, int* __restrict__ crowded,
                                                       int* __restrict__ ncrowded)
{
    __shared__ double l[3][kProjChunk], vx[kProjChunk], vy[kProjChunk];
    const int lane = threadIdx.x & 63, i = threadIdx.x >> 6;
    const int c0 = blockIdx.x * kProjCells, c = c0 + lane;
    const int s0 = c < nt ? start[c] : 0;
    int s1 = c < nt ? start[c + 1] : 0;
    const bool many = s1 - s0 > kProjMany;
    if (many) {
        if (i == 0) crowded[atomicAdd(ncrowded, 1)] = c;
        s1 = s0;
    }
    const bool some = __any(many);
    const int p0 = start[c0], p1 = start[min(c0 + kProjCells, nt)];
    double sx = 0.0, sy = 0.0, w = 0.0;
    for (int b = p0; b < p1; b += kProjChunk) {
        if (some) {   // on to the first particle of a cell that is summed here (every wave holds all the cells)
            int next = s1 > b && s0 < s1 ? max(s0, b) : p1;
#pragma unroll
            for (int off = 32; off > 0; off >>= 1) next = min(next, __shfl_xor(next, off, 64));
            b = next;
            if (b >= p1) break;
        }
        const int m = min(kProjChunk, p1 - b);
#pragma unroll
        for (int k = threadIdx.x; k < kProjChunk; k += kBlock)
            if (k < m) {
                const double2 l12 = lam12[b + k], v = vel[b + k];
                l[0][k] = l12.x;
                l[1][k] = l12.y;
                l[2][k] = lam3[b + k];
                vx[k] = v.x;
                vy[k] = v.y;
            }
        __syncthreads();
        if (i < 3) {
            const int k1 = min(s1, b + m) - b;
            for (int k = max(s0, b) - b; k < k1; ++k) {
                const double li = l[i][k];
                sx += li * vx[k];
                sy += li * vy[k];
                w += li;
            }
        }
        __syncthreads();
    }
    if (i < 3 && c < nt && !many) {
        double* o = part + 9 * (size_t)c + 3 * i;
        o[0] = sx;
        o[1] = sy;
        o[2] = w;
    }
}

// The listed cells, one to a wave: the particles pass through LDS, the next chunk's loads in flight, and nine lanes
// add one sum each, in array order (w as l_i times one). The chain of additions bounds it: 7 ns a particle of the
// largest cell.
constexpr int kCrowdChunk = 256, kCrowdBlocks = 2048;

__global__ __launch_bounds__(64) void k_proj_crowded(const int* __restrict__ ncrowded, const int* __restrict__ crowded,
                                                     const int* __restrict__ start, const double2* __restrict__ lam12,
                                                     const double* __restrict__ lam3, const double2* __restrict__ vel,
                                                     double* __restrict__ part)
{
    constexpr int R = kCrowdChunk / 64, kU = 8;
    __shared__ __align__(16) double l[3][kCrowdChunk], v[3][kCrowdChunk];
    const int lane = threadIdx.x, n = *ncrowded;
    for (int q = blockIdx.x; q < n; q += kCrowdBlocks) {
        const int c = crowded[q], s0 = start[c], s1 = start[c + 1];
        double2 l12[R], vv[R];
        double l3[R];
        auto fetch = [&](int b) {
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int p = min(b + lane + 64 * r, s1 - 1);
                l12[r] = lam12[p];
                l3[r] = lam3[p];
                vv[r] = vel[p];
            }
        };
        fetch(s0);
        double s = 0.0;
        for (int b = s0; b < s1; b += kCrowdChunk) {
            __syncthreads();
#pragma unroll
            for (int r = 0; r < R; ++r) {
                const int k = lane + 64 * r;
                l[0][k] = l12[r].x;
                l[1][k] = l12[r].y;
                l[2][k] = l3[r];
                v[0][k] = vv[r].x;
                v[1][k] = vv[r].y;
                v[2][k] = 1.0;
            }
            __syncthreads();
            if (b + kCrowdChunk < s1) fetch(b + kCrowdChunk);
            const int m = min(kCrowdChunk, s1 - b);
            if (lane < 9) {
                const double *lp = l[lane / 3], *vp = v[lane % 3];
                int k = 0;
                for (; k + kU <= m; k += kU) {
                    double t[kU];
#pragma unroll
                    for (int u = 0; u < kU; ++u) t[u] = lp[k + u] * vp[k + u];
#pragma unroll
                    for (int u = 0; u < kU; ++u) s += t[u];
                }
                for (; k < m; ++k) s += lp[k] * vp[k];
            }
        }
        if (lane < 9) part[9 * (size_t)c + lane] = s;
    }
}

__global__ void k_proj_nodes(int nv, const int* __restrict__ inc_off, const int* __restrict__ inc_code,
                             const double* __restrict__ part, double* __restrict__ u0, double* __restrict__ u1,
                             int* __restrict__ ncrowded)
{
    const int v = blockIdx.x * blockDim.x + threadIdx.x;
    if (v == 0) *ncrowded = 0;   // for the next projection
    if (v >= nv) return;
    double sx = 0.0, sy = 0.0, w = 0.0;
    for (int e = inc_off[v]; e < inc_off[v + 1]; ++e) {
        const int code = inc_code[e];
        const double* s = part + 9 * (size_t)(code >> 2) + 3 * (code & 3);
        sx += s[0];
        sy += s[1];
        w += s[2];
    }
    u0[v] = sx / w;
    u1[v] = sy / w;
}

// ------------------------------------------------------------------ host side
static void alloc_state(pfem_particles_t* ph, long cap)
{
    for (int b = 0; b < 2; ++b) {
        ph->cell[b].alloc(cap);
        ph->lam12[b].alloc(cap);
        ph->lam3[b].alloc(cap);
        ph->pos[b].alloc(cap);
        ph->vel[b].alloc(cap);
        ph->id[b].alloc(cap);
    }
    const size_t blocks = blocks_for(cap);
    ph->order.alloc(blocks * kBlock);    // (a range of kBlock per workgroup of k_advect)
    ph->order2.alloc(blocks * kBlock);
    ph->left_n.alloc(blocks);
    ph->tile_cell.alloc(cap / kTileOut + 2);
    ph->long_cells.alloc(cap / kLongCell + 1);
    ph->capacity = cap;
    ++ph->generation;
}

// The host copy of the device state {count, next ID, deleted, added}, once its pending copy is complete
// (normally long before: the stream has passed it by the next call that needs it).
static void sync_host_state(pfem_particles_t* ph)
{
    if (!ph->pst_pending) return;
    PFEM_HIP(hipEventSynchronize(ph->pst_ev));
    ph->count = ph->h_pst[0];
    ph->next_id = (uint32_t)ph->h_pst[1];
    ph->deleted_last = ph->h_pst[2];
    ph->added_last = ph->h_pst[3];
    ph->pst_pending = false;
}

// The device state from the host's (after a seed or an upload)
static void put_device_state(Context* c, pfem_particles_t* ph)
{
    ph->h_pst[0] = ph->count;
    ph->h_pst[1] = ph->next_id;
    ph->h_pst[2] = ph->deleted_last;
    ph->h_pst[3] = ph->added_last;
    h2d(c, ph->pst.p, ph->h_pst, 4 * sizeof(long));
    ph->pst_pending = false;
}

// capacity for `need` particles; the first ph->count particles of the current buffers are kept (the host
// state must be current)
static void grow(Context* c, pfem_particles_t* ph, long need)
{
    if (need <= ph->capacity) return;
    // deviceVector::resize grows by 1.1 (src/common/device_vector.cuh:96-109); keep more headroom
    const long cap = std::max<long>(need + need / 4, 1024);
    const int b = ph->cur;
    DevArray<int> cell(cap);
    DevArray<double2> l12(cap), pos(cap), vel(cap);
    DevArray<double> l3(cap);
    DevArray<uint32_t> id(cap);
    const size_t n = ph->count;
    PFEM_HIP(hipMemcpyAsync(cell.p, ph->cell[b].p, n * sizeof(int), hipMemcpyDeviceToDevice, c->stream));
    PFEM_HIP(hipMemcpyAsync(l12.p, ph->lam12[b].p, n * sizeof(double2), hipMemcpyDeviceToDevice, c->stream));
    PFEM_HIP(hipMemcpyAsync(l3.p, ph->lam3[b].p, n * sizeof(double), hipMemcpyDeviceToDevice, c->stream));
    PFEM_HIP(hipMemcpyAsync(pos.p, ph->pos[b].p, n * sizeof(double2), hipMemcpyDeviceToDevice, c->stream));
    PFEM_HIP(hipMemcpyAsync(vel.p, ph->vel[b].p, n * sizeof(double2), hipMemcpyDeviceToDevice, c->stream));
    PFEM_HIP(hipMemcpyAsync(id.p, ph->id[b].p, n * sizeof(uint32_t), hipMemcpyDeviceToDevice, c->stream));
    PFEM_HIP(hipStreamSynchronize(c->stream));
    alloc_state(ph, cap);
    ph->cell[b] = std::move(cell);
    ph->lam12[b] = std::move(l12);
    ph->lam3[b] = std::move(l3);
    ph->pos[b] = std::move(pos);
    ph->vel[b] = std::move(vel);
    ph->id[b] = std::move(id);
}

// cell_start of buffer b for the device count (grid over the capacity)
static void compute_cell_start(Context* c, pfem_particles_t* ph, int b)
{
    hipLaunchKernelGGL(k_cell_start, dim3(blocks_for(ph->capacity + 1)), dim3(kBlock), 0, c->stream,
                       (const long*)ph->pst.p, ph->cell[b].p, ph->mesh->nt, ph->cell_start.p);
}

static Centers centers_of(const pfem_particles_t* ph)
{
    Centers cen{};
    std::memcpy(cen.c, ph->centers, sizeof(cen.c));
    return cen;
}

// Host part of an advection step, before any launch: the count of the previous step, and capacity for
// the largest refill this step can make (every subcell of every cell). Never inside a captured region.
void particles_advect_prepare(pfem_particles_t* ph)
{
    Context* c = C(ph->ctx);
    pfem_mesh2d_t* m = ph->mesh;
    PFEM_REQUIRE(m->nbr_off.p, "the mesh was created without neighbour lists");
    sync_host_state(ph);
    grow(c, ph, ph->count + (long)m->nt * ph->ns);
}

// The launches of an advection step on buffer b (the particles end in buffer 1 - b): advection and
// relocation, census, refill, reorder by cell, the new device state and cell_start. Launches only (no
// host waits, allocations or host-side state), so that it can be captured; the caller sets ph->cur.
void particles_advect_launch(pfem_particles_t* ph, int b, const double* u0, const double* u1, double dt, int substeps)
{
    Context* c = C(ph->ctx);
    pfem_mesh2d_t* m = ph->mesh;
    const long cap = ph->capacity;
    const long* pst = ph->pst.p;
    const double dts = dt / substeps;
    const int nt = m->nt, tiles = (nt + kScanTile - 1) / kScanTile, o = 1 - b;
    const dim3 bl(kBlock), per_particle(blocks_for(cap)), per_cell(blocks_for(nt + 1));
    // mask, live and the counters are one array
    hipLaunchKernelGGL(k_zero_u32, dim3(blocks_for(2L * nt + 4)), bl, 0, c->stream, 2L * nt + 4, ph->mask.p);
    // (the places' arrays hold the lists of leaving particles until the places are known)
    hipLaunchKernelGGL(k_advect, per_particle, bl, 0, c->stream, pst, substeps, dts, (const int*)ph->cell[b].p,
                       ph->lam12[b].p, ph->lam3[b].p, ph->pos[b].p, m->tri.p, (const double4*)m->invJ.p, m->v3.p, u0, u1,
                       ph->level, 1.0 / ph->level, ph->mask.p, ph->live, ph->order.p, ph->order2.p, ph->left_n.p);
    auto relocate = [&](auto kernel, int particles) {   // of a workgroup
        hipLaunchKernelGGL(kernel, dim3(blocks_for(cap, particles)), bl, 0, c->stream, pst, substeps, dts,
                           ph->cell[b].p, ph->lam12[b].p, ph->lam3[b].p, ph->pos[b].p, m->tri.p,
                           (const double4*)m->invJ.p, m->v3.p, m->nbr_off.p, m->nbr_idx.p, u0, u1, ph->level,
                           1.0 / ph->level, ph->mask.p, ph->live, ph->order.p, ph->order2.p, ph->left_n.p, ph->counters);
    };
    // (256 CUs x 32 waves x 1024 particles: below, four lists a wave leave wave slots empty; and x 64 particles)
    if (cap >= (1L << 23)) relocate(k_relocate<4, 1>, 4 * kWaves * kBlock);
    else if (cap >= (1L << 19)) relocate(k_relocate<1, 1>, kWaves * kBlock);
    else relocate(k_relocate<1, kWaves>, kBlock);
    hipLaunchKernelGGL(k_cell_tiles, dim3(tiles), bl, 0, c->stream, nt, ph->ns, ph->mask.p, ph->live, ph->prefix.p,
                       ph->tile_sums.p);
    hipLaunchKernelGGL(k_cell_top, dim3(1), bl, 0, c->stream, tiles, ph->tile_sums.p, ph->counters, ph->pst.p);
    hipLaunchKernelGGL(k_cells, per_cell, bl, 0, c->stream, nt, pst, ph->live, ph->prefix.p, ph->tile_sums.p, ph->mask.p,
                       ph->ns, ph->cell_start.p, ph->cursor.p, ph->order.p, ph->tile_cell.p, ph->long_cells.p, ph->counters);
    hipLaunchKernelGGL(k_place, dim3(blocks_for(cap, kBlock * kPlaceRuns)), bl, 0, c->stream, pst, ph->cell[b].p,
                       ph->live, ph->cursor.p, ph->order.p, ph->order2.p);
    hipLaunchKernelGGL(k_order_long, dim3(kOrderBlocks), dim3(kOrderLanes), 0, c->stream, ph->counters, ph->long_cells.p,
                       ph->cell_start.p, ph->live, ph->order2.p, ph->order.p);
    hipLaunchKernelGGL(k_reorder, dim3(blocks_for(cap, kTileOut)), bl, 0, c->stream, ph->pst.p, ph->ns, ph->cell_start.p,
                       ph->live, ph->tile_cell.p, ph->order.p, ph->mask.p, ph->prefix.p, ph->tile_sums.p, m->xy.p, m->tri.p,
                       centers_of(ph), u0, u1, ph->cell[b].p, ph->lam12[b].p, ph->lam3[b].p, ph->pos[b].p, ph->vel[b].p,
                       ph->id[b].p, ph->cell[o].p, ph->lam12[o].p, ph->lam3[o].p, ph->pos[o].p, ph->vel[o].p, ph->id[o].p);
    hipLaunchKernelGGL(k_pstate_finish, dim3(1), dim3(64), 0, c->stream, ph->pst.p);
    PFEM_HIP(hipGetLastError());
}

// After the launches of a step: the device state's copy to the host, read at its next use
void particles_advect_post(pfem_particles_t* ph)
{
    Context* c = C(ph->ctx);
    PFEM_HIP(hipMemcpyAsync(ph->h_pst, ph->pst.p, 4 * sizeof(long), hipMemcpyDeviceToHost, c->stream));
    PFEM_HIP(hipEventRecord(ph->pst_ev, c->stream));
    ph->pst_pending = true;
}

void particles_advect(pfem_particles_t* ph, const double* u0, const double* u1, double dt, int substeps)
{
    PFEM_REQUIRE(substeps > 0, "substeps must be positive");
    particles_advect_prepare(ph);
    const int b = ph->cur;
    particles_advect_launch(ph, b, u0, u1, dt, substeps);
    ph->cur = 1 - b;
    particles_advect_post(ph);
}

void particles_project(pfem_particles_t* ph, double* u0, double* u1)
{
    Context* c = C(ph->ctx);
    pfem_mesh2d_t* m = ph->mesh;
    const int b = ph->cur;
    hipLaunchKernelGGL(k_proj_cells, dim3(blocks_for(m->nt, kProjCells)), dim3(kBlock), 0, c->stream, m->nt, ph->cell_start.p,
                       ph->lam12[b].p, ph->lam3[b].p, ph->vel[b].p, ph->part.p, ph->cursor.p, ph->counters + 3);
    hipLaunchKernelGGL(k_proj_crowded, dim3(kCrowdBlocks), dim3(64), 0, c->stream, ph->counters + 3, ph->cursor.p,
                       ph->cell_start.p, ph->lam12[b].p, ph->lam3[b].p, ph->vel[b].p, ph->part.p);
    hipLaunchKernelGGL(k_proj_nodes, dim3(blocks_for(m->nv)), dim3(kBlock), 0, c->stream, m->nv, m->inc.off.p,
                       m->inc.code.p, ph->part.p, u0, u1, ph->counters + 3);
    PFEM_HIP(hipGetLastError());
}

void particles_correct(pfem_particles_t* ph, const double* u0, const double* u1, const double* uo0, const double* uo1)
{
    Context* c = C(ph->ctx);
    const int b = ph->cur;
    hipLaunchKernelGGL(k_correct, dim3(blocks_for(ph->capacity)), dim3(kBlock), 0, c->stream, (const long*)ph->pst.p,
                       ph->cell[b].p, ph->lam12[b].p, ph->lam3[b].p, ph->vel[b].p, ph->mesh->tri.p, u0, u1, uo0,
                       uo1);
    PFEM_HIP(hipGetLastError());
}

// The particle set's buffer generation (changes when the buffers are reallocated) and current buffer
long particles_generation(const pfem_particles_t* ph) { return ph->generation; }
int particles_current(const pfem_particles_t* ph) { return ph->cur; }
void particles_set_current(pfem_particles_t* ph, int b) { ph->cur = b; }

}  // namespace pfem

using namespace pfem;

extern "C" {

// ParticleHandler2D constructor (particle_handler_2d.cu:238-294): level clamped to [1, 4], L^2 subcell
// centroids, row i from the top holding 2i+1 sub-triangles
int pfem_particles_create(pfem_mesh2d m, int level, pfem_particles* out)
{
    PFEM_TRY(m ? m->ctx : nullptr, {
        PFEM_REQUIRE(m && out, "null argument");
        auto ph = std::make_unique<pfem_particles_t>();
        ph->ctx = m->ctx;
        ph->mesh = m;
        const int L = std::max(std::min(level, 4), 1);
        ph->level = L;
        ph->ns = L * L;
        const double dx = 1.0 / L;
        int k = -1;
        for (int i = 0; i < L; ++i)
            for (int j = 0; j < 2 * i + 1; ++j) {
                const double xmin = (j / 2) * dx, xmax = xmin + dx;
                const double ymin = (L - 1 - i) * dx, ymax = ymin + dx;
                const double v0[3] = {xmin, ymax, 1.0 - xmin - ymax};
                double v1[3];
                v1[0] = (j % 2 == 0) ? xmin : xmax;
                v1[1] = (j % 2 == 0) ? ymin : ymax;
                v1[2] = 1.0 - v1[0] - v1[1];
                const double v2[3] = {xmax, ymin, 1.0 - xmax - ymin};
                ++k;
                for (int d = 0; d < 3; ++d) ph->centers[k][d] = (v0[d] + v1[d] + v2[d]) * 0.3333333333333333;
            }
        Context* c = C(m->ctx);
        ph->mask.alloc(2 * (size_t)m->nt + 4);
        ph->live = (int*)ph->mask.p + m->nt;
        ph->counters = ph->live + m->nt;
        ph->cursor.alloc(m->nt + 1);
        ph->prefix.alloc(m->nt + 1);
        ph->tile_sums.alloc(m->nt / kScanTile + 1);
        ph->cell_start.alloc(m->nt + 1);
        ph->part.alloc(9 * (size_t)m->nt);
        ph->pst.alloc(8);
        PFEM_HIP(hipHostMalloc((void**)&ph->h_pst, 4 * sizeof(long), hipHostMallocDefault));
        PFEM_HIP(hipEventCreateWithFlags(&ph->pst_ev, hipEventDisableTiming));
        zero_async(c, ph->mask.p, ph->mask.bytes());
        alloc_state(ph.get(), 1024);
        put_device_state(c, ph.get());
        zero_async(c, ph->cell_start.p, ph->cell_start.bytes());   // no particles: every cell's range is empty
        PFEM_HIP(hipStreamSynchronize(c->stream));
        *out = ph.release();
    });
}

int pfem_particles_destroy(pfem_particles ph)
{
    if (!ph) return PFEM_OK;
    (void)hipStreamSynchronize(ph->ctx->stream);
    delete ph;
    return PFEM_OK;
}

int pfem_particles_seed(pfem_particles ph, int mode, int ppc, uint64_t seed)
{
    PFEM_TRY(ph ? ph->ctx : nullptr, {
        PFEM_REQUIRE(ph, "null argument");
        PFEM_REQUIRE(mode == 0 || mode == 1, "seed mode must be 0 (subcell centroids) or 1 (random)");
        if (mode == 0) ppc = ph->ns;
        PFEM_REQUIRE(ppc > 0, "particles per cell must be positive");
        Context* c = C(ph->ctx);
        const long P = (long)ph->mesh->nt * ppc;
        sync_host_state(ph);
        ph->count = 0;
        grow(c, ph, P + P / 5);
        const int b = ph->cur;
        const uint2 key = make_uint2((uint32_t)seed, (uint32_t)(seed >> 32));
        hipLaunchKernelGGL(k_seed, dim3(blocks_for(P)), dim3(kBlock), 0, c->stream, ph->mesh->nt, ppc, mode,
                           ph->mesh->xy.p, ph->mesh->tri.p, centers_of(ph), key, ph->cell[b].p, ph->lam12[b].p,
                           ph->lam3[b].p, ph->pos[b].p, ph->vel[b].p, ph->id[b].p);
        PFEM_HIP(hipGetLastError());
        ph->count = P;
        ph->next_id = (uint32_t)P;
        ph->deleted_last = ph->added_last = 0;
        put_device_state(c, ph);
        compute_cell_start(c, ph, b);
        PFEM_HIP(hipStreamSynchronize(c->stream));
    });
}

int pfem_particles_init_velocity(pfem_particles ph, const double* d_u0, const double* d_u1)
{
    PFEM_TRY(ph ? ph->ctx : nullptr, {
        PFEM_REQUIRE(ph && d_u0 && d_u1, "null argument");
        particles_correct(ph, d_u0, d_u1, nullptr, nullptr);
    });
}

int pfem_particles_advect(pfem_particles ph, const double* d_u0, const double* d_u1, double dt, int substeps)
{
    PFEM_TRY(ph ? ph->ctx : nullptr, {
        PFEM_REQUIRE(ph && d_u0 && d_u1, "null argument");
        particles_advect(ph, d_u0, d_u1, dt, substeps);
    });
}

int pfem_particles_project(pfem_particles ph, double* d_u0, double* d_u1)
{
    PFEM_TRY(ph ? ph->ctx : nullptr, {
        PFEM_REQUIRE(ph && d_u0 && d_u1, "null argument");
        particles_project(ph, d_u0, d_u1);
    });
}

int pfem_particles_correct(pfem_particles ph, const double* d_u0, const double* d_u1, const double* d_uo0,
                           const double* d_uo1)
{
    PFEM_TRY(ph ? ph->ctx : nullptr, {
        PFEM_REQUIRE(ph && d_u0 && d_u1 && d_uo0 && d_uo1, "null argument");
        particles_correct(ph, d_u0, d_u1, d_uo0, d_uo1);
    });
}

int pfem_particles_count(pfem_particles ph, long* count)
{
    PFEM_TRY(ph ? ph->ctx : nullptr, {
        PFEM_REQUIRE(ph && count, "null argument");
        sync_host_state(ph);
        *count = ph->count;
    });
}

int pfem_particles_download(pfem_particles ph, int* cell, double* lam, double* pos, double* vel, uint32_t* id)
{
    PFEM_TRY(ph ? ph->ctx : nullptr, {
        PFEM_REQUIRE(ph, "null argument");
        Context* c = C(ph->ctx);
        sync_host_state(ph);
        const size_t n = ph->count;
        const int b = ph->cur;
        if (cell) d2h_sync(c, cell, ph->cell[b].p, n * sizeof(int));
        if (lam) {
            std::vector<double2> l12(n);
            std::vector<double> l3(n);
            d2h_sync(c, l12.data(), ph->lam12[b].p, n * sizeof(double2));
            d2h_sync(c, l3.data(), ph->lam3[b].p, n * sizeof(double));
            for (size_t p = 0; p < n; ++p) {
                lam[3 * p] = l12[p].x;
                lam[3 * p + 1] = l12[p].y;
                lam[3 * p + 2] = l3[p];
            }
        }
        if (pos) d2h_sync(c, pos, ph->pos[b].p, n * sizeof(double2));
        if (vel) d2h_sync(c, vel, ph->vel[b].p, n * sizeof(double2));
        if (id) d2h_sync(c, id, ph->id[b].p, n * sizeof(uint32_t));
    });
}

int pfem_particles_upload(pfem_particles ph, long count, const int* cell, const double* lam, const double* pos,
                          const double* vel, const uint32_t* id, uint32_t next_id)
{
    PFEM_TRY(ph ? ph->ctx : nullptr, {
        PFEM_REQUIRE(ph && count >= 0 && cell && lam && pos && vel && id, "null argument");
        for (long p = 0; p < count; ++p) {
            PFEM_REQUIRE(cell[p] >= 0 && cell[p] < ph->mesh->nt, "particle cell out of range");
            PFEM_REQUIRE(p == 0 || cell[p] >= cell[p - 1], "uploaded particles must be ordered by cell");
        }
        Context* c = C(ph->ctx);
        sync_host_state(ph);
        ph->count = 0;
        grow(c, ph, count + count / 5 + 16);
        const int b = ph->cur;
        std::vector<double2> l12(count);
        std::vector<double> l3(count);
        for (long p = 0; p < count; ++p) {
            l12[p] = make_double2(lam[3 * p], lam[3 * p + 1]);
            l3[p] = lam[3 * p + 2];
        }
        h2d(c, ph->cell[b].p, cell, count * sizeof(int));
        h2d(c, ph->lam12[b].p, l12.data(), count * sizeof(double2));
        h2d(c, ph->lam3[b].p, l3.data(), count * sizeof(double));
        h2d(c, ph->pos[b].p, pos, count * sizeof(double2));
        h2d(c, ph->vel[b].p, vel, count * sizeof(double2));
        h2d(c, ph->id[b].p, id, count * sizeof(uint32_t));
        ph->count = count;
        ph->next_id = next_id;
        ph->deleted_last = ph->added_last = 0;
        put_device_state(c, ph);
        compute_cell_start(c, ph, b);
        PFEM_HIP(hipStreamSynchronize(c->stream));
    });
}

int pfem_particles_stats(pfem_particles ph, long* deleted_last, long* added_last)
{
    PFEM_TRY(ph ? ph->ctx : nullptr, {
        PFEM_REQUIRE(ph, "null argument");
        sync_host_state(ph);
        if (deleted_last) *deleted_last = ph->deleted_last;
        if (added_last) *added_last = ph->added_last;
    });
}

}  // extern "C"
