// Resident PCG: a whole Jacobi (or unpreconditioned) PCG solve as one launch.
//
// What bounds the launch-per-kernel PCG of a system of up to a few 100k rows is not its bytes (they stay in
// the caches) but three launches and their chains of dependent loads per iteration: 14.5 us at 4k to 40k
// rows, against about 1 us for the arithmetic. Here a workgroup of 1024 lanes owns 1024
// rows for the whole solve, one row per lane: the row's matrix entries and r live in its
// registers, p (own rows and halo), x and the diagonal in LDS, and nothing is streamed per iteration. Two
// things cross workgroups:
//   * the halo: z is published row by row into one of three rotating buffers whose unpublished
//     locations read as the sentinel NaN of sync.hpp. p at the halo columns is kept by the reader (p = z +
//     beta p, as its owner computes it), and z is published before beta is known, so the exchange runs
//     under the reduction that yields beta;
//   * the two sums of an iteration: every 256-row tile publishes its partial into a slot, and every
//     workgroup adds all slots in the order the launch-per-kernel path uses (sum_partials), so alpha,
//     beta, the iterates and the iteration count are those of that path, bit for bit.
// Measured on MI355X: publish to visible in a polling workgroup 0.52 us; a sum over 16, 80 and 256 slots
// 1.2, 2.3 and 2.7 us; an iteration 1.8 us at 1k rows (one workgroup), 3.7 at 4k, 5.5 at 40k, 9.0 at 251k.
//
// Ordering without fences (an agent-scope fence would write back and invalidate the XCD's L2): all shared
// values are written with agent-scope stores, which go through to the point of coherence, and a
// workgroup waits for its own stores (s_waitcnt) before it publishes its next partial. A buffer or slot is
// re-armed with the sentinel only after a sum that every reader contributed to following its last read,
// and is polled again only after a later sum; hence no reader can see a stale value.
//
// Progress: a workgroup waits for others of its system, so they must be resident together. The host
// launches only grids (single solve) or systems (batch: systems in dispatch order, so the earliest
// unfinished system is always complete or next in line) that fit the device. If other work holds the
// device for too long, a wait exceeds its poll limit, the launch ends with an error flag and the caller
// solves with the launch-per-kernel path instead.
#include <algorithm>
#include <climits>
#include <condition_variable>
#include <mutex>

#include "device.hpp"
#include "internal.hpp"
#include "resident.hpp"
#include "solver.hpp"
#include "resident_wait.hpp"

namespace pfem {

constexpr int kResLanes = 1024;            // rows and lanes of a workgroup
constexpr int kResTiles = kResLanes / kBlock;
constexpr int kResHalo = 2 * kResLanes;    // halo columns a workgroup can hold (two per lane)
constexpr int kResTable = 4096;            // hash table for the halo's columns

template <typename T>
struct ResArgs {
    int nsys;                // systems; workgroups [sys[k].blk0, sys[k + 1].blk0) solve system k
    const ResSys* sys;
    const int* rowptr;
    const int* col;
    const T* val;
    const T* invd;
    const T* b;
    T* x;
    const int* tiles;        // SpMV tile table (single system; its order is the (p, Ap) slots'), or null
    void* zbuf;              // 3 n values of T
    unsigned long long* ring;   // 4 x all tiles
    long nz;                 // n
    int nt;                  // all tiles
    ResOut* out;
    int* err;                // 1: a wait failed, 2: a halo does not fit
    long limit;              // polls of one wait
    double tol;
    int tol_mode, maxit, x_zero;
    double drop;             // reliable updates: replacement after gamma fell by this factor
};

__device__ __forceinline__ unsigned res_hash(int c) { return ((unsigned)c * 2654435761u) >> 20; }   // 12 bits

// Column c into the hash table; false if that is full
__device__ __forceinline__ bool res_insert(int* key, int c)
{
    unsigned h = res_hash(c);
#pragma unroll 1
    for (int tries = 0; tries < kResTable; ++tries) {
        const int old = atomicCAS(&key[h], -1, c);
        if (old == -1 || old == c) return true;
        h = (h + 1) & (kResTable - 1);
    }
    return false;
}

// The system of a workgroup
__device__ __forceinline__ int res_system(int nsys, const ResSys* __restrict__ sys, int block)
{
    int lo = 0, hi = nsys - 1;
    while (lo < hi) {
        const int mid = (lo + hi + 1) >> 1;
        if (sys[mid].blk0 <= block) lo = mid;
        else hi = mid - 1;
    }
    return lo;
}

// For a batch's plan: sets *over if a workgroup's rows use more columns of others than it can hold
__global__ __launch_bounds__(kResLanes) void k_resident_halo(int nsys, const ResSys* __restrict__ sys,
                                                             const int* __restrict__ rowptr, const int* __restrict__ col,
                                                             int* __restrict__ over)
{
    __shared__ int key[kResTable];
    __shared__ int halo;
    const int tid = threadIdx.x;
    const ResSys S = sys[res_system(nsys, sys, blockIdx.x)];
    const int first = S.row0 + ((int)blockIdx.x - S.blk0) * kResLanes, last = min(first + kResLanes, S.row0 + S.rows);
    for (int k = tid; k < kResTable; k += kResLanes) key[k] = -1;
    if (tid == 0) halo = 0;
    __syncthreads();
    bool fits = true;
    if (first + tid < last)
        for (int k = rowptr[first + tid]; k < rowptr[first + tid + 1]; ++k)
            if (col[k] < first || col[k] >= last) fits &= res_insert(key, col[k]);
    __syncthreads();
    int n = fits ? 0 : kResTable;
    for (int k = tid; k < kResTable; k += kResLanes) n += key[k] >= 0;
    if (n) atomicAdd(&halo, n);
    __syncthreads();
    if (tid == 0 && halo > kResHalo) *over = 1;
}

struct ResShared {
    double wave[2 * (kResLanes / 64)];   // wave sums
    double total[kWaves];
    int slot[kResTiles];           // slots of the workgroup's tiles in the (p, Ap) sums
    int from[kResTiles];           // a single workgroup: the tile of each of those slots
    int fail, halo;
};

// Sum of v over the system's rows, in the order of block_partials and sum_partials; every lane gets it.
// e counts the sums of the solve (which of the four slot sets). All lanes call it; the waves that do not
// collect slots run meanwhile().
template <typename T, typename F>
__device__ __forceinline__ double res_sum(const ResArgs<T>& a, const ResSys& S, int blk, int nblk, int e, bool permuted,
                                          double v, ResShared& sh, F&& meanwhile)
{
    using U = unsigned long long;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    v = wave_sum(v);
    if (nblk == 1) {
        // at most four tiles, whose sums are at lanes 0, 4, 8, 12; the slots' sum is (t0 + t2) + (t1 + t3)
        double* w = sh.wave + (e & 1) * (kResLanes / 64);   // alternating, so one barrier is enough
        if (lane == 0) w[wid] = v;
        __syncthreads();
        const int k = lane & 15;
        const double t = sum4(w[permuted ? kWaves * sh.from[k >> 2] + (k & 3) : k]);
        const double q = t + lane_down<8>(t);
        return uniform(q + lane_down<4>(q));
    }
    if (lane == 0) sh.wave[wid] = v;
    asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // this lane's published and re-armed values are visible
    __syncthreads();
    U* ring = a.ring + (size_t)(e & 3) * a.nt + S.tile0;
    const int t0 = blk * kResTiles;
    if (tid < 16 && t0 + tid / kWaves < S.ntiles) {
        const double t = sum4(sh.wave[tid]);
        if ((tid & 3) == 0) {
            const int slot = permuted ? sh.slot[tid / kWaves] : t0 + tid / kWaves;
            publish(reinterpret_cast<double*>(ring) + slot, t);
            __hip_atomic_store(a.ring + (size_t)((e + 2) & 3) * a.nt + S.tile0 + slot, Sentinel<double>::bits,
                               __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
    }
    if (wid < kWaves) {
        double s = 0.0;
        for (int k = tid; k < S.ntiles; k += kBlock)
            s += res_await<double>(ring + k, __hip_atomic_load(ring + k, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                                   a.err, a.limit, &sh.fail);
        s = wave_sum(s);
        if (lane == 0) sh.total[wid] = s;
    } else {
        meanwhile();
    }
    __syncthreads();
    return uniform(sum4(sh.total[lane & 3]));
}

// REL: reliable updates (batched PFEM_PRECISION_MIXED): the iterations run in FP64 like everything here, and
// the true residual b - A x replaces the recursive one after every fall of gamma by `drop` and for the
// stopping test.
// WPS waves per SIMD: 4 is one workgroup to a CU; 8 holds two (with 6 vector and up to 16 scalar registers spilled:
// 10% slower alone), so that in a batch of more workgroups than CUs one team's waits are another's work. With REL
// it is 24 to 31 and 26, and a mixed batch takes 13 to 18% longer than an FP64 one (15.1 and 17.0 ms for 64 systems).
template <typename T, int W, bool JAC, bool REL, int WPS>
__global__ __launch_bounds__(kResLanes, WPS) void k_resident_cg(ResArgs<T> a)
{
    using U = typename Sentinel<T>::U;
    constexpr U sent = Sentinel<T>::bits;
    // the hash table and the list of halo columns are needed only before p is
    constexpr int kTableBytes = kResTable * 4 + kResTable * 2 + kResHalo * 4;
    constexpr int kVecBytes = (kResLanes + kResHalo + 1) * (int)sizeof(T);   // own rows, halo, a zero
    __shared__ __align__(16) char lds[kTableBytes > kVecBytes ? kTableBytes : kVecBytes];
    __shared__ ResShared sh;
    __shared__ T xl[kResLanes];               // x, read and written once an iteration by its own lane
    __shared__ T dl[JAC ? kResLanes : 1];     // the Jacobi diagonal
    T* pl = reinterpret_cast<T*>(lds);
    const int tid = threadIdx.x;

    const int lo = res_system(a.nsys, a.sys, blockIdx.x);
    const ResSys S = a.sys[lo];
    const int nblk = (S.rows + kResLanes - 1) / kResLanes;
    const int blk = (int)blockIdx.x - S.blk0;
    const int first = S.row0 + blk * kResLanes, last = min(first + kResLanes, S.row0 + S.rows);
    const int row = first + tid;
    const bool on = row < last;

    // ---- the row's entries; columns of other workgroups become halo slots through a hash table
    int* key = reinterpret_cast<int*>(lds);
    unsigned short* idx = reinterpret_cast<unsigned short*>(lds + kResTable * 4);
    int* list = reinterpret_cast<int*>(lds + kResTable * 4 + kResTable * 2);
    for (int k = tid; k < kResTable; k += kResLanes) key[k] = -1;
    if (tid == 0) sh.fail = sh.halo = 0;
    __syncthreads();
    const int k0 = on ? a.rowptr[row] : 0, len = on ? a.rowptr[row + 1] - k0 : 0;
#pragma unroll 1
    for (int e = 0; e < len; ++e) {
        const int c = a.col[k0 + e];
        if (c >= first && c < last) continue;
        if (!res_insert(key, c)) sh.halo = kResTable;
    }
    __syncthreads();
    for (int k = tid; k < kResTable; k += kResLanes)
        if (key[k] >= 0) {
            const int i = atomicAdd(&sh.halo, 1);
            idx[k] = (unsigned short)i;
            if (i < kResHalo) list[i] = key[k];
        }
    __syncthreads();
    const int halo = sh.halo;
    if (halo > kResHalo) {   // this pattern does not fit: nobody waits for this workgroup for long
        if (tid == 0) __hip_atomic_fetch_max(a.err, 2, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        return;
    }
    // the entries' places in LDS as byte offsets, two to a register; unused entries take the zero (s + 0 * 0)
    unsigned cw[W / 2];
#pragma unroll
    for (int e = 0; e < W; ++e) {
        int at = kResLanes + kResHalo;
        if (e < len) {
            const int c = a.col[k0 + e];
            at = c - first;
            if (c < first || c >= last) {
                unsigned h = res_hash(c);
#pragma unroll 1
                while (key[h] != c) h = (h + 1) & (kResTable - 1);
                at = kResLanes + idx[h];
            }
        }
        at *= (int)sizeof(T);
        if (e & 1) cw[e / 2] |= (unsigned)at << 16;
        else cw[e / 2] = (unsigned)at;
    }
    T av[W];
#pragma unroll
    for (int e = 0; e < W; ++e) av[e] = e < len ? a.val[k0 + e] : (T)0;
    // the halo columns of this lane; the first 768 go to the waves that collect no slots in res_sum
    auto hidx = [&](int u) { return ((tid + kResLanes - kBlock) & (kResLanes - 1)) + u * kResLanes; };
    constexpr unsigned kNone = ~0u;
    unsigned hc[2];   // byte offsets: one base address in scalar registers serves all lanes
#pragma unroll
    for (int u = 0; u < 2; ++u) {
        hc[u] = hidx(u) < halo ? (unsigned)list[hidx(u)] * (unsigned)sizeof(T) : kNone;
    }
    if (tid < kResTiles) {
        const int t = blk * kResTiles + tid;
        sh.slot[tid] = t;
        if (a.tiles && t < S.ntiles)   // the slot whose tile starts at this tile's first row
            for (int s = 0; s < S.ntiles; ++s)
                if (a.tiles[2 * s] == first + tid * kBlock) sh.slot[tid] = s;
        if (nblk == 1) sh.from[t < S.ntiles ? sh.slot[tid] : tid] = tid;
    }
    __syncthreads();

    if (tid == 0) pl[kResLanes + kResHalo] = 0;
    auto product = [&]() {   // the row of A times the vector in LDS, entries in CSR order
        T s = 0;
#pragma unroll
        for (int e = 0; e < W; ++e)
            s += av[e] * *reinterpret_cast<const T*>(lds + ((e & 1) ? cw[e / 2] >> 16 : cw[e / 2] & 0xFFFFu));
        return s;
    };
    char* const zb = reinterpret_cast<char*>(a.zbuf);
    const size_t zbytes = sizeof(T) * (size_t)a.nz;
    const unsigned at = (unsigned)row * (unsigned)sizeof(T);
    // Exchange i uses buffer i mod 3 and re-arms the next one's, last read in exchange i - 2: every reader has
    // contributed to a sum since. (With two buffers, the exchange of x below would re-arm the buffer of the z
    // published just before it, which another workgroup may still be reading.)
    int ex = 0;
    auto next = [&]() { ex = ex == 2 ? 0 : ex + 1; };
    auto offer = [&](T v) {   // publish this row's value of the current exchange
        if (nblk > 1 && on) {
            publish(reinterpret_cast<T*>(zb + ex * zbytes + at), v);
            __hip_atomic_store(reinterpret_cast<U*>(zb + (ex == 2 ? 0 : ex + 1) * zbytes + at), sent, __ATOMIC_RELAXED,
                               __HIP_MEMORY_SCOPE_AGENT);
        }
    };
    T hv[2] = {0, 0};
    auto take = [&]() {      // the halo's values of the current exchange
        U v[2] = {0, 0};
        char* const q = zb + ex * zbytes;
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (hc[u] != kNone) v[u] = __hip_atomic_load(reinterpret_cast<U*>(q + hc[u]), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (hc[u] != kNone) hv[u] = res_await<T>(reinterpret_cast<U*>(q + hc[u]), v[u], a.err, a.limit, &sh.fail);
    };
    auto nothing = [] {};
    const bool collects = tid < kBlock;

    // ---- r = b - A x, z = M^-1 r, p = z
    T r = on ? a.b[row] : (T)0;
    if (JAC) dl[tid] = on ? a.invd[row] : (T)1;
    xl[tid] = on && !a.x_zero ? a.x[row] : (T)0;
    double bmb = (double)(JAC ? r * (r * dl[tid]) : r * r);
    if (!a.x_zero) {
        pl[tid] = xl[tid];
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (hc[u] != kNone) pl[kResLanes + hidx(u)] = a.x[hc[u] / (unsigned)sizeof(T)];
        __syncthreads();
        r = r - product();
    }
    auto prec = [&]() { return JAC ? r * dl[tid] : r; };   // z, recomputed where it is needed
    offer(prec());
    int e = 0;
    const bool perm = !a.x_zero;
    double gam = res_sum(a, S, blk, nblk, e++, perm, on ? (double)(r * prec()) : 0.0, sh, nothing);
    bmb = a.x_zero ? gam : res_sum(a, S, blk, nblk, e++, perm, on ? bmb : 0.0, sh, nothing);
    const double thr = a.tol_mode == PFEM_TOL_RELATIVE && bmb > 0.0 ? a.tol * a.tol * bmb : a.tol * a.tol;
    double gend = gam, gmax = gam;   // the last gamma the stopping test saw
    int it = 0, nrep = 0;
    bool nan = gam != gam, converged = gam < thr;
    bool done = nan || converged;
    if (!done) take();
#pragma unroll
    for (int u = 0; u < 2; ++u)
        if (hc[u] != kNone) pl[kResLanes + hidx(u)] = hv[u];
    pl[tid] = prec();
    __syncthreads();
    while (!done && !sh.fail) {
        const T q = product();
        const double pq = res_sum(a, S, blk, nblk, e++, true, on ? (double)(pl[tid] * q) : 0.0, sh, nothing);
        if (sh.fail) break;
        const T alpha = (T)(gam / pq);
        xl[tid] += alpha * pl[tid];
        r = r - alpha * q;
        next();
        offer(prec());
        double g = res_sum(a, S, blk, nblk, e++, false, on ? (double)(r * prec()) : 0.0, sh, take);
        if (sh.fail) break;
        ++it;
        bool taken = !collects;
        if (!REL) {
            gend = g;
            nan = g != g;
            converged = !nan && g < thr;
            done = nan || converged || it >= a.maxit;
        } else {
            nan = g != g;
            done = nan || it >= a.maxit;
            if (!done && (g < thr || g < a.drop * gmax)) {
                // r = b - A x: x takes p's place in LDS meanwhile
                next();
                offer(xl[tid]);
                take();
                const T p = pl[tid];
                T ph[2] = {0, 0};
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    if (hc[u] != kNone) ph[u] = pl[kResLanes + hidx(u)];
                pl[tid] = xl[tid];
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    if (hc[u] != kNone) pl[kResLanes + hidx(u)] = hv[u];
                __syncthreads();
                if (sh.fail) break;
                r = (on ? a.b[row] : (T)0) - product();
                __syncthreads();
                pl[tid] = p;
#pragma unroll
                for (int u = 0; u < 2; ++u)
                    if (hc[u] != kNone) pl[kResLanes + hidx(u)] = ph[u];
                g = res_sum(a, S, blk, nblk, e++, false, on ? (double)(r * prec()) : 0.0, sh, nothing);
                if (sh.fail) break;
                next();     // re-arms the buffer of the z above: only now has every workgroup read it
                offer(prec());
                taken = false;
                ++nrep;
                gend = g;
                nan = g != g;
                converged = !nan && g < thr;
                done = nan || converged;
                gmax = g;
            }
        }
        if (done) break;
        const T beta = (T)(g / gam);
        gam = g;
        if (!taken) take();
        pl[tid] = prec() + beta * pl[tid];
#pragma unroll
        for (int u = 0; u < 2; ++u)
            if (hc[u] != kNone) pl[kResLanes + hidx(u)] = hv[u] + beta * pl[kResLanes + hidx(u)];
        __syncthreads();
    }
    if (sh.fail) return;
    if (on) a.x[row] = xl[tid];
    if (blk == 0 && tid == 0) {
        ResOut& o = a.out[lo];
        o.it = it;
        o.converged = converged;
        o.nan = nan;
        o.nrep = nrep;
        o.res = sqrt(fabs(gend));
        o.tdone = wall_clock64();
    }
}

// Sentinels in the exchange buffers and the slots, cleared results, the start of the clock, and the initial
// guess kept for a launch that has to be given up
template <typename T>
__global__ void k_resident_prepare(long nz, typename Sentinel<T>::U* __restrict__ zb, long nr,
                                   unsigned long long* __restrict__ ring, int nsys, ResOut* __restrict__ out,
                                   int* __restrict__ err, long n, const T* __restrict__ x, T* __restrict__ keep)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) keep[i] = x[i];
    if (i < nz) zb[i] = Sentinel<T>::bits;
    if (i < nr) ring[i] = Sentinel<double>::bits;
    if (i < nsys) {
        out[i] = ResOut{};
        out[i].t0 = wall_clock64();
    }
    if (i == 0) *err = 0;
}

namespace {
template <typename T>
using Kernel = void (*)(ResArgs<T>);

template <typename T, int W, int WPS>
Kernel<T> kernel_of(bool jac, bool rel)
{
    if constexpr (sizeof(T) == 8)
        if (rel) return jac ? k_resident_cg<T, W, true, true, WPS> : k_resident_cg<T, W, false, true, WPS>;
    return jac ? k_resident_cg<T, W, true, false, WPS> : k_resident_cg<T, W, false, false, WPS>;
}

template <typename T>
Kernel<T> kernel_for(int width, bool jac, bool rel, bool two_per_cu)
{
    if (width > 8) return kernel_of<T, 16, 4>(jac, rel);
    if constexpr (sizeof(T) == 8)
        if (two_per_cu) return kernel_of<T, 8, 8>(jac, rel);
    return kernel_of<T, 8, 4>(jac, rel);
}
}  // namespace

namespace {
struct Seats {
    std::mutex m;
    std::condition_variable freed;
    int used = 0;
    unsigned long next = 0, serving = 0;   // tickets
};
Seats& seats(int device)
{
    static Seats s[64];
    return s[device & 63];
}
}  // namespace

ResidentSeats::ResidentSeats(int device, int blocks, int cus)
    : device_(device), taken_(std::min((blocks + 7) / 8 * 8, cus))
{
    Seats& s = seats(device_);
    std::unique_lock<std::mutex> lock(s.m);
    const unsigned long ticket = s.next++;
    s.freed.wait(lock, [&] { return s.serving == ticket && s.used + taken_ <= cus; });
    s.used += taken_;
    ++s.serving;
    s.freed.notify_all();
}

ResidentSeats::~ResidentSeats()
{
    Seats& s = seats(device_);
    std::lock_guard<std::mutex> lock(s.m);
    s.used -= taken_;
    s.freed.notify_all();
}

int resident_blocks(int rows) { return (rows + kResLanes - 1) / kResLanes; }

bool ResidentWork::plan(Context* c, std::shared_ptr<Pattern> p, const std::vector<int>& rows, bool single)
{
    // 262144 rows: the launch-per-kernel path adds one partial per 256 rows up to there. Every SpMV tile must
    // hold 256 rows (a tile also ends at 2048 non-zeros: 3D matrices), or its sums are grouped differently.
    constexpr int kMaxRows = 1024 * kBlock, kMaxWidth = 16;
    if (pat == p && sys_rows == rows && tiles_permuted == single) return fits;
    pause = 0;
    tiles_permuted = single;
    pat = std::move(p);
    sys_rows = rows;
    fits = false;
    const Pattern& P = *pat;
    width = 0;
    for (int i = 0; i < P.n; ++i) width = std::max(width, P.h_rowptr[i + 1] - P.h_rowptr[i]);
    if (width > kMaxWidth) return false;
    nsys = (int)rows.size() - 1;
    order.resize(nsys);
    for (int k = 0; k < nsys; ++k) order[k] = k;
    std::stable_sort(order.begin(), order.end(),
                     [&](int u, int v) { return rows[u + 1] - rows[u] > rows[v + 1] - rows[v]; });
    std::vector<ResSys> h(nsys);
    blocks = tiles = largest = 0;
    for (int q = 0; q < nsys; ++q) {
        const int k = order[q], nr = rows[k + 1] - rows[k];
        if (nr < 1 || nr > kMaxRows) return false;
        const int nt = (nr + kBlock - 1) / kBlock;
        for (int t = 0; t < nt; ++t) {
            const int r0 = rows[k] + t * kBlock, r1 = std::min(r0 + kBlock, rows[k + 1]);
            if (P.h_rowptr[r1] - P.h_rowptr[r0] > kResTileNnz) return false;
        }
        h[q] = ResSys{rows[k], nr, tiles, nt, blocks};
        tiles += nt;
        blocks += resident_blocks(nr);
        largest = std::max(largest, resident_blocks(nr));
    }
    upload(c, sys, h);
    err.alloc(1);
    if (!single) {
        // A halo that does not fit ends a single system's first launch; in a batch the other systems would be solved
        // in vain, so the halos are counted first (0.28 ms for 14.8M rows; on the host 0.9 ms for 262144).
        zero_async(c, err.p, sizeof(int));
        hipLaunchKernelGGL(k_resident_halo, dim3(blocks), dim3(kResLanes), 0, c->stream, nsys, sys.p, P.rowptr.p, P.col.p,
                           err.p);
        PFEM_HIP(hipGetLastError());
        int over = 0;
        d2h_sync(c, &over, err.p, sizeof(int));
        if (over) return false;
    }
    ring.alloc(4 * (size_t)tiles);
    zbuf.alloc(4 * (size_t)P.n);   // three exchange buffers and the initial guess
    out.alloc(nsys);
    if (h_out) (void)hipHostFree(h_out);
    h_out = nullptr;
    PFEM_HIP(hipHostMalloc((void**)&h_out, sizeof(ResOut) * nsys + sizeof(int), hipHostMallocDefault));
    fits = true;
    return true;
}

ResidentWork::~ResidentWork()
{
    if (h_out) (void)hipHostFree(h_out);
}

template <typename T>
bool ResidentWork::solve(Context* c, const T* val, const T* invd, const T* b, T* x, bool x_zero, double tol, int tol_mode,
                         int maxit, double drop, int spin_limit)
{
    if (!fits) return false;
    if (pause > 0) {
        --pause;
        return false;
    }
    const bool rel = drop > 0.0;
    int per_cu = 0, cus = 0;
    PFEM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device));
    Kernel<T> k = kernel_for<T>(width, invd != nullptr, rel, blocks > cus);
    PFEM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)k, kResLanes, 0));
    if (largest > per_cu * cus) return false;
    const Pattern& P = *pat;
    ResArgs<T> a{};
    a.nsys = nsys;
    a.sys = sys.p;
    a.rowptr = P.rowptr.p;
    a.col = P.col.p;
    a.val = val;
    a.invd = invd;
    a.b = b;
    a.x = x;
    a.tiles = tiles_permuted ? P.tiles.p : nullptr;
    a.zbuf = zbuf.p;
    a.ring = reinterpret_cast<unsigned long long*>(ring.p);
    a.nz = P.n;
    a.nt = tiles;
    a.out = out.p;
    a.err = err.p;
    // At the default of 65536 and about 1.1 us a poll: 18 ms for one system, whose workgroups start together
    // unless other work holds the device; 0.6 s for a batch, whose next system in line waits for a whole
    // solve to end.
    a.limit = nsys == 1 ? spin_limit / 4 : 8L * spin_limit;
    a.tol = tol;
    a.tol_mode = tol_mode;
    a.maxit = maxit;
    a.x_zero = x_zero ? 1 : 0;
    a.drop = drop;
    T* keep = reinterpret_cast<T*>(zbuf.p) + 3 * (size_t)P.n;
    const ResidentSeats held(c->device, blocks, cus);
    const long nfill = std::max({3L * P.n, 4L * tiles, (long)nsys});
    hipLaunchKernelGGL(k_resident_prepare<T>, dim3(blocks_for(nfill)), dim3(kBlock), 0, c->stream, 3L * P.n,
                       reinterpret_cast<typename Sentinel<T>::U*>(zbuf.p), 4L * tiles, a.ring, nsys, out.p, err.p,
                       x_zero ? 0L : (long)P.n, (const T*)x, keep);
    hipLaunchKernelGGL(k, dim3(blocks), dim3(kResLanes), 0, c->stream, a);
    PFEM_HIP(hipGetLastError());
    int* h_err = reinterpret_cast<int*>(h_out + nsys);
    PFEM_HIP(hipMemcpyAsync(h_out, out.p, sizeof(ResOut) * nsys, hipMemcpyDeviceToHost, c->stream));
    PFEM_HIP(hipMemcpyAsync(h_err, err.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    PFEM_HIP(hipStreamSynchronize(c->stream));
    if (*h_err == 0) return true;
    if (*h_err == 2) {
        fits = false;   // a halo that never fits
    } else {
        ++given_up;
        if (spin_limit > 0) pause = kResPause;
    }
    if (!x_zero) PFEM_HIP(hipMemcpyAsync(x, keep, sizeof(T) * (size_t)P.n, hipMemcpyDeviceToDevice, c->stream));
    return false;
}

template bool ResidentWork::solve<double>(Context*, const double*, const double*, const double*, double*, bool, double,
                                          int, int, double, int);
template bool ResidentWork::solve<float>(Context*, const float*, const float*, const float*, float*, bool, double, int,
                                         int, double, int);

void ResidentWorkDeleter::operator()(ResidentWork* w) const { delete w; }

}  // namespace pfem
