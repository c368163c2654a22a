// Resident IC0-PCG: the iterations of a PCG solve with a multicolour IC0 factor as one launch.
//
// What bounds the launch-per-kernel iteration (SpMV, forward and backward sweep) of a system of up to a few
// 100k rows is the chain of its waits: three launches, each a tail and a start over, and a colour's rows waiting
// for those of the one before through chunks of 512 rows that lie anywhere in the mesh. Here a workgroup of 1024
// lanes owns a compact patch of up to 1024 nodes for the whole solve, one row of the factor's ordering per lane:
// the row's entries of A and of L, x and r live in its registers, p and the sweeps' values of the patch and of
// its halo in LDS, and nothing is streamed per iteration. Colour by colour the lanes of a colour finish their rows
// from LDS; only rows on a patch's rim are published for the patches beside it, whose lanes wait for them into
// their halo places before the next colour. An iteration's chain is then one exchange per colour and sweep and
// one sum over the workgroups: (y, y) = (r, M^-1 r) is published after the forward sweep and read after the
// backward one, so only (p, A p) is waited for.
//
// Rows of 9 to 12 neighbours have a variant of their own that spills 25 of those registers: 16.0, 16.7, 18.0 and 19.1 us
// an iteration at 5k, 13k, 65k and 256k rows, against 23.4, 22.9, 21.9 and 30.8 launch by launch.
//
// us per iteration at 13k, 65k, 132k and 256k rows: 26.0, 25.5, 26.7 and 31.4 launch by launch, 11.4, 12.5, 12.9 and
// 13.5 here: 0.6 for the product, about 2.5 for (p, A p), 1.2 for each of the sweeps' eight steps (0.52 of it a
// published value's way). Looking four times as often for a value came out slower (13.8), and so did halo places on
// lanes whose wave publishes nothing meanwhile (12.9); values scattered over the vector instead of packed by patch
// took 14.8.
//
// Ordering without fences, as in resident.hip: shared values go through to the point of coherence, places that
// are not published yet read as a sentinel NaN. The y and z of an iteration have one of two buffers in turn.
// The other one, last read before the (p, A p) sum of this iteration, is re-armed after it and before this
// workgroup's part of (y, y), which every workgroup has read before it polls that buffer again.
//
// Progress: all workgroups must be resident together, which the host checks. If other work holds the device for
// too long a wait exceeds its poll limit, the launch ends with an error flag and the caller goes on with the
// launch-per-kernel iterations from the start it had prepared.
#include <algorithm>
#include <cmath>
#include <numeric>

#include "device.hpp"
#include "internal.hpp"
#include "quotient.hpp"
#include "resident_ic0.hpp"
#include "resident_wait.hpp"

namespace pfem {

constexpr int kIcLanes = 1024;          // rows, halo rows and lanes of a workgroup
constexpr int kIcMaxBlocks = 256;       // one ring slot per lane of four waves
constexpr int kIcNoColour = 255;

template <typename TS>
struct IcArgs {
    const int *rows, *halo, *steps;
    const int *post, *from;         // exchange places: of a rim row (or -1), of a halo row
    const uint32_t *info, *hinfo;   // rows: colour | lower entries << 9 | entries << 15; halo: colour | wanted forward << 8
    const uint16_t* slot;
    const int* rowptr;
    const double* aval;
    const int *lptr, *uptr;         // the split factor's row offsets
    const TS* f;
    const TS* d;
    const double* scale;            // scale[1] = c^2 of a 16-bit factor, or null
    const double *x, *r, *p;
    double* xo;
    double *yb, *zb;                // two buffers of n places each
    unsigned long long* ring;       // four sets of a slot per workgroup
    long n;                         // exchange places
    const CgState* st;
    CgState* out;
    int* err;
    long limit;
};

struct IcShared {
    double wave[kIcLanes / 64], total[kWaves], one[2];
    int fail;
};

// Sum over the workgroup's lanes of v, published as this workgroup's part of sum e
__device__ __forceinline__ void ic_offer(unsigned long long* ring, int e, double v, IcShared& sh)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nb = gridDim.x;
    v = wave_sum(v);
    if (lane == 0) sh.wave[wid] = v;
    __syncthreads();
    if (wid == 0) {
        const double t = wave_sum(lane < kIcLanes / 64 ? sh.wave[lane] : 0.0);
        if (lane == 0) {
            if (nb == 1) {
                sh.one[e & 1] = t;
            } else {
                publish(reinterpret_cast<double*>(ring) + (e & 3) * nb + blockIdx.x, t);
                __hip_atomic_store(ring + ((e + 2) & 3) * nb + blockIdx.x, Sentinel<double>::bits, __ATOMIC_RELAXED,
                                   __HIP_MEMORY_SCOPE_AGENT);
            }
        }
    }
}

// Sum e, in every lane; v: the caller's first look at its slot
__device__ __forceinline__ unsigned long long ic_look(unsigned long long* ring, int e)
{
    const int nb = gridDim.x;
    return nb > 1 && (int)threadIdx.x < nb ? __hip_atomic_load(ring + (e & 3) * nb + threadIdx.x, __ATOMIC_RELAXED,
                                                               __HIP_MEMORY_SCOPE_AGENT)
                                           : 0ull;
}

__device__ __forceinline__ double ic_sum(unsigned long long* ring, int e, unsigned long long v, int* err, long limit,
                                         IcShared& sh)
{
    const int lane = threadIdx.x & 63, wid = threadIdx.x >> 6, nb = gridDim.x;
    if (nb > 1 && wid < kWaves) {
        double s = 0.0;
        if ((int)threadIdx.x < nb) s = res_await<double>(ring + (e & 3) * nb + threadIdx.x, v, err, limit, &sh.fail);
        s = wave_sum(s);
        if (lane == 0) sh.total[wid] = s;
    }
    __syncthreads();
    return nb == 1 ? sh.one[e & 1] : uniform(sum4(sh.total[lane & 3]));
}

template <typename TS, int W>
__global__ __launch_bounds__(kIcLanes, 4) void k_resident_ic0(IcArgs<TS> a)
{
    using SF = typename std::conditional<sizeof(TS) == 8, double, float>::type;   // holds the factor's values exactly
    constexpr int kZero = 2 * kIcLanes;
    __shared__ double pl[2 * kIcLanes + 1], yl[2 * kIcLanes + 1];   // own rows, halo, a zero
    __shared__ IcShared sh;
    const int tid = threadIdx.x;
    const size_t lanes = (size_t)gridDim.x * kIcLanes, g = (size_t)blockIdx.x * kIcLanes + tid;
    const int row = a.rows[g], hrow = a.halo[g], steps = a.steps[blockIdx.x];
    const int post = a.post[g], from = a.from[g];
    const bool on = row >= 0;
    const unsigned info = a.info[g], hinfo = a.hinfo[g];
    const int colour = info & 255, len = (info >> 15) & 63;
    int nl = (info >> 9) & 63;
    const int hcolour = hinfo & 255;
    const bool rim = post >= 0, hforward = (hinfo >> 8) & 1;
    if (tid == 0) {
        sh.fail = 0;
        pl[kZero] = yl[kZero] = 0.0;
    }
    unsigned cw[W / 2];   // places of the entries as byte offsets, two to a register
    double av[W], ad = 0.0, ld = 1.0, li = 1.0;
    SF lv[W];
    const int k0 = on ? a.rowptr[row] : 0, kl = on ? a.lptr[row] : 0, ku = on ? a.uptr[row] : 0;
#pragma unroll
    for (int e = 0; e < W; ++e) {
        const unsigned at = 8u * (e < len ? a.slot[e * lanes + g] : kZero);
        if (e & 1) cw[e / 2] |= at << 16;
        else cw[e / 2] = at;
        av[e] = e < len ? a.aval[k0 + e + (e >= nl ? 1 : 0)] : 0.0;
        lv[e] = e < len ? (SF)a.f[e < nl ? kl + e : ku + e - nl] : (SF)0;
    }
    double x = 0.0, r = 0.0, p0 = 0.0;
    if (on) {
        ad = a.aval[k0 + nl];
        ld = (double)a.d[row];
        li = 1.0 / ld;
        x = a.x[row];
        r = a.r[row];
        p0 = a.p[row];
    }
    pl[tid] = p0;
    pl[kIcLanes + tid] = hrow >= 0 ? a.p[hrow] : 0.0;
    yl[tid] = yl[kIcLanes + tid] = 0.0;
    const double c2 = sizeof(TS) == 2 ? a.scale[1] : 1.0;
    double gam = a.st->gam[0], res = a.st->res;
    const double thr = a.st->thr;
    const int maxit = a.st->maxit;
    int it = 0, done = a.st->done, nan = a.st->nan, converged = a.st->converged;
    auto place = [&](const double* v, int e) {
        return *reinterpret_cast<const double*>(reinterpret_cast<const char*>(v) + ((e & 1) ? cw[e / 2] >> 16 : cw[e / 2] & 0xFFFFu));
    };
    int e = 0;
    __syncthreads();
    while (!done) {
        asm volatile("" : "+v"(nl));   // the entries' tests stay in the loop: kept across it their masks spill
        double q = ad * pl[tid];   // A p
#pragma unroll
        for (int k = 0; k < W; ++k) q += av[k] * place(pl, k);
        ic_offer(a.ring, e, on ? pl[tid] * q : 0.0, sh);
        const double pq = ic_sum(a.ring, e, ic_look(a.ring, e), a.err, a.limit, sh);
        ++e;
        if (sh.fail) return;
        const double alpha = gam / pq;
        x += alpha * pl[tid];
        r = r - alpha * q;
        double* const yb = a.yb + (it & 1) * a.n;
        double* const zb = a.zb + (it & 1) * a.n;
        if (rim) {
            unsigned long long* const y1 = reinterpret_cast<unsigned long long*>(a.yb + ((it + 1) & 1) * a.n);
            unsigned long long* const z1 = reinterpret_cast<unsigned long long*>(a.zb + ((it + 1) & 1) * a.n);
            __hip_atomic_store(y1 + post, Sentinel<double>::bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
            __hip_atomic_store(z1 + post, Sentinel<double>::bits, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
        // y = L^-1 r, colour by colour
        double y = 0.0;
        for (int c = 0; c < steps; ++c) {
            if (c == colour) {
                double s = sizeof(TS) == 2 ? r * c2 : r;
#pragma unroll
                for (int k = 0; k < W; ++k)
                    s -= (k < nl ? (double)lv[k] : 0.0) * place(yl, k);
                y = quotient_near(s, ld, li);
                yl[tid] = y;
                if (rim) publish(yb + post, y);
            }
            if (c == hcolour && hforward) {
                unsigned long long* const at = reinterpret_cast<unsigned long long*>(yb + from);
                yl[kIcLanes + tid] = res_await<double>(at, __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                                                       a.err, a.limit, &sh.fail);
            }
            __syncthreads();
        }
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");   // the re-armed places are visible
        ic_offer(a.ring, e, y * y, sh);
        // z = L^-T y, in y's place
        unsigned long long v = 0;
        for (int c = steps - 1; c >= 0; --c) {
            if (c == colour) {
                double s = y;
#pragma unroll
                for (int k = 0; k < W; ++k)
                    s -= (k < nl ? 0.0 : (double)lv[k]) * place(yl, k);
                y = quotient_near(s, ld, li);
                yl[tid] = y;
                if (rim) publish(zb + post, y);
            }
            if (c == 0) v = ic_look(a.ring, e);
            if (c == hcolour) {
                unsigned long long* const at = reinterpret_cast<unsigned long long*>(zb + from);
                yl[kIcLanes + tid] = res_await<double>(at, __hip_atomic_load(at, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT),
                                                       a.err, a.limit, &sh.fail);
            }
            __syncthreads();
        }
        double gnew = ic_sum(a.ring, e, v, a.err, a.limit, sh);
        ++e;
        if (sh.fail) return;
        if (sizeof(TS) == 2) gnew /= c2;
        // the end of the iteration, as cg_record
        ++it;
        res = sqrt(fabs(gnew));
        nan = gnew != gnew;
        converged = !nan && gnew < thr;
        done = nan || converged || it >= maxit;
        const double beta = gnew / gam;
        gam = gnew;
        pl[tid] = yl[tid] + beta * pl[tid];
        pl[kIcLanes + tid] = hrow >= 0 ? yl[kIcLanes + tid] + beta * pl[kIcLanes + tid] : 0.0;
        __syncthreads();
    }
    if (on) a.xo[row] = x;
    if (blockIdx.x == 0 && tid == 0) {
        CgState o = *a.st;
        o.gam[it & 1] = gam;
        o.it = it;
        o.res = res;
        o.done = done;
        o.nan = nan;
        o.converged = converged;
        *a.out = o;
    }
}

__global__ void k_ic0_arm(long n, unsigned long long* __restrict__ buf, int nr, unsigned long long* __restrict__ ring,
                          int* __restrict__ err)
{
    const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (i < n) buf[i] = Sentinel<double>::bits;
    if (i < nr) ring[i] = Sentinel<double>::bits;
    if (i == 0) *err = 0;
}

ResidentIc0::~ResidentIc0()
{
    if (h_err) (void)hipHostFree(h_err);
}

// The nodes `in` (marked by mark[v] == id) in breadth-first order from a node far from the others; levels: how
// many there are
static void spread(const Pattern& P, std::vector<int>& mark, int id, std::vector<int>& in, int& levels)
{
    std::vector<int> out;
    out.reserve(in.size());
    int seed = in[0];
    for (int pass = 0; pass < 2; ++pass) {   // the last node reached from any one is far out
        const int seen = -(id + 2 + pass);
        for (int v : in) mark[v] = id;
        out.clear();
        levels = 0;
        size_t next = 0;
        for (size_t head = 0, end = 0; out.size() < in.size(); ) {
            if (head == out.size()) {        // another component
                if (!out.empty() || pass == 0) while (mark[in[next]] != id) ++next;
                const int s = out.empty() ? seed : in[next];
                mark[s] = seen;
                out.push_back(s);
            }
            end = out.size();
            ++levels;
            for (; head < end; ++head)
                for (int k = P.h_rowptr[out[head]]; k < P.h_rowptr[out[head] + 1]; ++k) {
                    const int w = P.h_col[k];
                    if (mark[w] == id) {
                        mark[w] = seen;
                        out.push_back(w);
                    }
                }
        }
        seed = out.back();
    }
    in.swap(out);
}

bool ResidentIc0::plan(Context* c, const pfem_precond_t* pc)
{
    if (pat == pc->fpat && colours == pc->h_lptr) return fits;
    pat = pc->fpat;
    colours = pc->h_lptr;
    fits = false;
    pause = 0;
    const Pattern& P = *pat;
    const int n = P.n, nc = (int)colours.size() - 1;
    if (n < 1 || n > kIcLanes * kIcMaxBlocks || nc < 1 || nc >= kIcNoColour || colours[0] != 0 || colours[nc] != n) return false;
    std::vector<int> colour(n);
    for (int k = 0; k < nc; ++k)
        for (int i = colours[k]; i < colours[k + 1]; ++i) colour[i] = k;
    int most = 0;
    for (int i = 0; i < n; ++i) {
        bool diag = false;
        for (int k = P.h_rowptr[i]; k < P.h_rowptr[i + 1]; ++k) {
            const int j = P.h_col[k];
            if (j == i) diag = true;
            else if ((j < i) != (colour[j] < colour[i]) || colour[j] == colour[i]) return false;
        }
        if (!diag) return false;
        most = std::max(most, P.h_rowptr[i + 1] - P.h_rowptr[i] - 1);
    }
    if (most > 12) return false;   // the entries of a row are a lane's registers
    width = most <= 8 ? 8 : 12;
    // Patches: the nodes in breadth-first order cut into strips about as wide as a square patch, each strip in
    // breadth-first order along itself cut into patches.
    blocks = (n + kIcLanes - 1) / kIcLanes;
    std::vector<int> order(n), mark(n, -1);
    std::iota(order.begin(), order.end(), 0);
    int id = 0, levels = 1;
    if (blocks > 1) {
        spread(P, mark, id, order, levels);
        id += 4;
        const double side = std::sqrt((double)n / blocks);
        const int strips = std::max(1, std::min(blocks, (int)std::lround(levels / side)));
        for (int s = 0; s < strips; ++s) {
            const long b0 = (long)blocks * s / strips, b1 = (long)blocks * (s + 1) / strips;
            const long v0 = (long)n * b0 / blocks, v1 = (long)n * b1 / blocks;
            if (b1 - b0 < 2) continue;
            std::vector<int> in(order.begin() + v0, order.begin() + v1);
            int l;
            for (int v : in) mark[v] = id;
            spread(P, mark, id, in, l);
            id += 4;
            std::copy(in.begin(), in.end(), order.begin() + v0);
        }
    }
    const size_t lanes = (size_t)blocks * kIcLanes;
    std::vector<int> h_rows(lanes, -1), h_halo(lanes, -1), h_steps(blocks, 0), block(n), at(n);
    std::vector<int> h_post(lanes, -1), h_from(lanes, -1);
    std::vector<uint32_t> h_info(lanes, (uint32_t)kIcNoColour), h_hinfo(lanes, (uint32_t)kIcNoColour);
    std::vector<uint16_t> h_slot((size_t)width * lanes, 0);
    for (int b = 0; b < blocks; ++b) {
        const long v0 = (long)n * b / blocks, v1 = (long)n * (b + 1) / blocks;
        std::sort(order.begin() + v0, order.begin() + v1);   // rows ascend: colour by colour
        for (long v = v0; v < v1; ++v) {
            block[order[v]] = b;
            at[order[v]] = (int)(v - v0);
            h_rows[(size_t)b * kIcLanes + (v - v0)] = order[v];
        }
    }
    places = 0;
    std::vector<int> where(n, -1), hs;   // halo place of a row in the block under work
    for (int b = 0; b < blocks; ++b) {
        const size_t l0 = (size_t)b * kIcLanes;
        hs.clear();
        for (int t = 0; t < kIcLanes && h_rows[l0 + t] >= 0; ++t) {
            const int i = h_rows[l0 + t];
            for (int k = P.h_rowptr[i]; k < P.h_rowptr[i + 1]; ++k)
                if (block[P.h_col[k]] != b && where[P.h_col[k]] < 0) {
                    where[P.h_col[k]] = 0;
                    hs.push_back(P.h_col[k]);
                }
        }
        if (hs.size() > (size_t)kIcLanes) return false;
        std::sort(hs.begin(), hs.end());
        for (size_t u = 0; u < hs.size(); ++u) {
            where[hs[u]] = (int)u;
            h_halo[l0 + u] = hs[u];
            h_hinfo[l0 + u] = (uint32_t)colour[hs[u]];
            h_steps[b] = std::max(h_steps[b], colour[hs[u]] + 1);
        }
        for (int t = 0; t < kIcLanes && h_rows[l0 + t] >= 0; ++t) {
            const int i = h_rows[l0 + t];
            int nl = 0, e = 0, rim = 0;
            for (int k = P.h_rowptr[i]; k < P.h_rowptr[i + 1]; ++k) {
                const int j = P.h_col[k];
                if (j == i) continue;
                const bool own = block[j] == b;
                nl += j < i;
                rim |= !own;   // the pattern is symmetric: a neighbour in another patch has this row in its halo
                if (!own && j < i) h_hinfo[l0 + where[j]] |= 256u;
                h_slot[(size_t)e++ * lanes + l0 + t] = (uint16_t)(own ? at[j] : kIcLanes + where[j]);
            }
            if (rim) h_post[l0 + t] = places++;
            h_info[l0 + t] = (uint32_t)colour[i] | (uint32_t)nl << 9 | (uint32_t)e << 15;
            h_steps[b] = std::max(h_steps[b], colour[i] + 1);
        }
        for (int j : hs) where[j] = -1;
        places = (places + 15) / 16 * 16;   // a patch's places start a cache line
    }
    // an unsymmetric pattern would leave a halo row unpublished
    for (size_t l = 0; l < lanes; ++l)
        if (h_halo[l] >= 0) {
            h_from[l] = h_post[(size_t)block[h_halo[l]] * kIcLanes + at[h_halo[l]]];
            if (h_from[l] < 0) return false;
        }
    upload(c, rows, h_rows);
    upload(c, halo, h_halo);
    upload(c, steps, h_steps);
    upload(c, post, h_post);
    upload(c, from, h_from);
    upload(c, info, h_info);
    upload(c, hinfo, h_hinfo);
    upload(c, slot, h_slot);
    buf.alloc(4 * (size_t)places + n);   // two y, two z, the solution
    ring.alloc(4 * (size_t)blocks);
    out.alloc(1);
    err.alloc(1);
    if (!h_err) PFEM_HIP(hipHostMalloc((void**)&h_err, sizeof(int), hipHostMallocDefault));
    fits = true;
    return true;
}

template <typename TS>
static void launch(Context* c, ResidentIc0& w, pfem_precond_t* pc, const TS* f, const double* scale, const double* x,
                   const double* r, const double* p, const CgState* st)
{
    const Pattern& P = *w.pat;
    auto k = w.width == 8 ? k_resident_ic0<TS, 8> : k_resident_ic0<TS, 12>;
    IcArgs<TS> a{};
    a.rows = w.rows.p;
    a.halo = w.halo.p;
    a.steps = w.steps.p;
    a.post = w.post.p;
    a.from = w.from.p;
    a.info = w.info.p;
    a.hinfo = w.hinfo.p;
    a.slot = w.slot.p;
    a.rowptr = P.rowptr.p;
    a.aval = pc->aval.p;
    a.lptr = pc->split_ptr.p;
    a.uptr = pc->split_ptr.p + (P.n + 1);
    a.f = f;
    a.d = f + pc->split_diag;
    a.scale = scale;
    a.x = x;
    a.r = r;
    a.p = p;
    a.yb = w.buf.p;
    a.zb = w.buf.p + 2 * (size_t)w.places;
    a.xo = w.buf.p + 4 * (size_t)w.places;
    a.ring = reinterpret_cast<unsigned long long*>(w.ring.p);
    a.n = w.places;
    a.st = st;
    a.out = w.out.p;
    a.err = w.err.p;
    // 0.6 s at the default of 65536 and about 1.1 us a poll: other work on the device may hold back some of the
    // workgroups, and the launch-per-kernel path's sums are grouped differently (other last bits)
    a.limit = 8L * pc->spin_limit;
    const long nfill = std::max({4L * w.places, 4L * w.blocks, 1L});
    hipLaunchKernelGGL(k_ic0_arm, dim3(blocks_for(nfill)), dim3(kBlock), 0, c->stream, 4L * w.places,
                       reinterpret_cast<unsigned long long*>(w.buf.p), 4 * w.blocks, a.ring, w.err.p);
    hipLaunchKernelGGL(k, dim3(w.blocks), dim3(kIcLanes), 0, c->stream, a);
    PFEM_HIP(hipGetLastError());
}

template <typename TS>
static bool fits_device(const ResidentIc0& w, int cus)
{
    auto k = w.width == 8 ? k_resident_ic0<TS, 8> : k_resident_ic0<TS, 12>;
    int per_cu = 0;
    PFEM_HIP(hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, (const void*)k, kIcLanes, 0));
    return w.blocks <= per_cu * cus;
}

bool ResidentIc0::solve(Context* c, pfem_precond_t* pc, bool reduced, double* x, const double* r, const double* p,
                        const CgState* st, CgState* hst)
{
    if (!fits) return false;
    if (pause > 0) {
        --pause;
        return false;
    }
    const bool half = reduced && pc->factor_bits == 16 && pc->half_ok;
    int cus = 0;
    PFEM_HIP(hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, c->device));
    if (!(half ? fits_device<_Float16>(*this, cus) : reduced ? fits_device<float>(*this, cus) : fits_device<double>(*this, cus)))
        return false;
    const ResidentSeats held(c->device, blocks, cus);
    if (half) launch<_Float16>(c, *this, pc, pc->split16.p, pc->scale16.p, x, r, p, st);
    else if (reduced) launch<float>(c, *this, pc, pc->split32.p, nullptr, x, r, p, st);
    else launch<double>(c, *this, pc, pc->split.p, nullptr, x, r, p, st);
    PFEM_HIP(hipMemcpyAsync(hst, out.p, sizeof(CgState), hipMemcpyDeviceToHost, c->stream));
    PFEM_HIP(hipMemcpyAsync(h_err, err.p, sizeof(int), hipMemcpyDeviceToHost, c->stream));
    PFEM_HIP(hipStreamSynchronize(c->stream));
    if (*h_err) {
        ++given_up;
        if (pc->spin_limit > 0) pause = kResPause;
        return false;
    }
    PFEM_HIP(hipMemcpyAsync(x, buf.p + 4 * (size_t)places, sizeof(double) * (size_t)pat->n, hipMemcpyDeviceToDevice, c->stream));
    return true;
}

void ResidentIc0Deleter::operator()(ResidentIc0* w) const { delete w; }

}  // namespace pfem
