// Band sweeps: the IC0/ILU0 triangular solves of a factor whose dependency levels are many and small -- the
// natural ordering of a structured mesh (401 levels of about 100 rows at 40k rows).
//
// What bounds such a solve is its chain of levels. The chunked sweeps (precond.hip) pass every value from
// workgroup to workgroup through memory, about 1.6 us a level: 615 + 668 us an apply at 40k rows. Here a
// workgroup takes a band of up to 8192 consecutive rows, holds their values in LDS, and ONE of its waves
// solves the band level by level: rows of a level sit on the wave's lanes, a dependency is an LDS read
// of what the same wave wrote, and no barrier is needed. The wave's matrix entries come in slices laid out
// in the order it takes them and are loaded eight slices ahead into registers. Only values of other bands
// cross workgroups: two waves poll them where their bands publish them and put them into LDS, in the order
// of their use, ahead of the solving wave, and one wave publishes the band's own (the sentinel protocol
// of sync.hpp; bands wait only on bands dispatched before them). Bands follow each other down the level
// chain a few levels behind. A quotient by the diagonal is formed from its reciprocal and two corrections, which gives the
// correctly rounded quotient (Markstein, "IA-64 and Elementary Functions", 2000) at a third of the
// division's latency, so results are those of the sequential solve, bit for bit. A level takes 0.15 us.
//
// Measured (MI355X, FP64 IC0 apply, chunked sweeps -> here): unit square 40k rows, 401 levels 1292 -> 147 us,
// 160k rows, 801 levels 4227 -> 321 us; cylinder 1M rows, 2689 levels 30.6 -> 1.64 ms; 3D box 133k rows, 151
// levels 1299 -> 187 us; tridiagonal, 8192 levels 13.2 -> 2.35 ms.
#include <algorithm>
#include <cmath>

#include "band.hpp"
#include "device.hpp"
#include "sync.hpp"

namespace pfem {

constexpr int kBandRows = 8192;    // 64 KB of values
constexpr int kBandHalo = 4096;    // values of other bands a band can hold: a mesh line or two

template <typename TV, typename TS, typename TF>
struct BandArgs {
    int n, rows;
    const int *soff, *hoff, *halo, *ooff, *out_at;
    const char* data;
    const TV* src;
    TV* out;
    TF *sy, *sw;
    double* part;
    const int* done;
    int* err;
    int limit;
};

// Bytes of a slice's planes, and where each begins
template <int W, typename TS>
struct SlicePlanes {
    static constexpr int diag = 64 * W * (int)sizeof(TS);
    static constexpr int place = diag + 1024;
    static constexpr int row = place + 256 * W;
    static constexpr int bytes = row + 256;
};

// What a lane needs of one slice, in registers
template <int W, typename TS>
struct BandSlot {
    TS v[W];
    unsigned at[W], row;   // byte offsets into LDS
    double d, ri;
};

template <int W, typename TS, bool UNIT>
__device__ __forceinline__ void band_load(BandSlot<W, TS>& t, const char* __restrict__ p, unsigned lane)
{
    using P = SlicePlanes<W, TS>;
    constexpr int per = 16 / (int)sizeof(TS);
    struct alignas(16) Values { TS v[per]; };
#pragma unroll
    for (int k = 0; k < W / per; ++k) {
        const Values q = *reinterpret_cast<const Values*>(p + 1024 * k + 16u * lane);
#pragma unroll
        for (int u = 0; u < per; ++u) t.v[k * per + u] = q.v[u];
    }
#pragma unroll
    for (int k = 0; k < W / 4; ++k) {
        const uint4 q = *reinterpret_cast<const uint4*>(p + P::place + 1024 * k + 16u * lane);
        t.at[4 * k] = q.x;
        t.at[4 * k + 1] = q.y;
        t.at[4 * k + 2] = q.z;
        t.at[4 * k + 3] = q.w;
    }
    t.row = *reinterpret_cast<const unsigned*>(p + P::row + 4u * lane);
    if (!UNIT) {
        const double2 q = *reinterpret_cast<const double2*>(p + P::diag + 16u * lane);
        t.d = q.x;
        t.ri = q.y;
    }
}

// s / d from ri = 1 / d (correctly rounded): the first quotient is within two units in the last place, the
// second within one, and Markstein's theorem makes the third the correctly rounded one as long as no step
// under- or overflows: |d| in [2^-100, 2^100] (else ri is stored as a NaN) and |q| >= 2^-800 or s = 0. A
// result outside (NaNs included) is formed again by the division.
__device__ __forceinline__ double quotient(double s, double d, double ri)
{
    const double q0 = s * ri;
    const double q1 = fma(fma(-d, q0, s), ri, q0);
    return __builtin_copysign(fma(fma(-d, q1, s), ri, q1), q0);   // (the sign of a zero)
}
__device__ __forceinline__ bool quotient_ok(double q) { return fabs(q) >= 0x1p-800 || q == 0.0; }
__device__ __forceinline__ float quotient(float s, float d, double) { return s / d; }
__device__ __forceinline__ bool quotient_ok(float q) { return q == q; }

// A value in LDS: 8 bytes for FP32 too, so that places are the same byte offsets
template <typename TF>
struct alignas(8) BandCell {
    TF v;
};

// UPPER: backward solve (values z into sw, initial values y from sy); UNIT: no division. D slices are in
// flight. LDS: the band's values, the halo's, a zero, a slot for idle lanes.
template <typename TV, typename TS, typename TF, int W, bool UPPER, bool UNIT>
__global__ __launch_bounds__(kBlock, 1) void k_band_sweep(BandArgs<TV, TS, TF> a)
{
    using U = typename Sentinel<TF>::U;
    constexpr U sent = Sentinel<TF>::bits;
    constexpr int D = W <= 8 ? 8 : 4;
    __shared__ BandCell<TF> y[kBandRows + kBandHalo + 2];
    __shared__ int solved;   // slices the solving wave has finished
    if (a.done && *a.done) return;
    const int tid = threadIdx.x, lane = tid & 63, wid = tid >> 6;
    const int band = UPPER ? (int)(gridDim.x - 1 - blockIdx.x) : (int)blockIdx.x;
    const int r0 = band * a.rows, cnt = min(a.rows, a.n - r0);
    const int h0 = a.hoff[band], nh = a.hoff[band + 1] - h0;
    for (int i = tid; i < cnt; i += kBlock) {
        if constexpr (UPPER) {
            y[i].v = a.sy[r0 + i];
            a.sy[r0 + i] = sentinel_value<TF>();   // re-armed for the next forward sweep
        } else {
            y[i].v = (TF)a.src[r0 + i];
            a.sw[r0 + i] = sentinel_value<TF>();
        }
    }
    for (int h = tid; h < nh; h += kBlock) y[kBandRows + h].v = sentinel_value<TF>();
    if (tid < 2) y[kBandRows + kBandHalo + tid].v = (TF)tid;   // a zero for unused entries, a one for idle lanes
    if (tid == 0) solved = 0;
    __syncthreads();
    TF* const mine = UPPER ? a.sw : a.sy;
    auto cell = [&](unsigned at) { return reinterpret_cast<U*>(reinterpret_cast<char*>(y) + at); };
    if (wid == kWaves - 1) {
        // publishes the values that other bands wait for, as soon as they are solved (the solving wave would
        // have to wait for its stores before it may use the loads it issues after them)
        const int o1 = a.ooff[band + 1];
        for (int o = a.ooff[band] + lane; o < o1; o += 64) {
            const int row = a.out_at[2 * o], slice = a.out_at[2 * o + 1];
            // each lane acts inside the loop: after it, every value would wait for the last lane's
            for (bool open = true; __any(open);) {
                if (open && __hip_atomic_load(&solved, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP) > slice) {
                    publish(mine + r0 + row, __builtin_bit_cast(TF, __hip_atomic_load(cell(8u * row), __ATOMIC_RELAXED,
                                                                                      __HIP_MEMORY_SCOPE_WORKGROUP)));
                    open = false;
                }
            }
        }
    } else if (wid > 0) {
        // The halo in the order of its first use, 64 values to a wave. All bands that fit the device start at once,
        // so the wait of a band for its first value spans the chains of all bands before it: up to 8192 levels
        // of 0.15 to 0.24 us each, 2 ms, for which it has another quarter of the limit, about 7 ms at the default.
        const long limit = a.limit + (long)(a.limit / 4) * blockIdx.x;
        for (int h = tid - 64; h < nh; h += kBlock - 128) {
            U* const q = reinterpret_cast<U*>(mine + a.halo[h0 + h]);
            long spins = 0;
            for (bool open = true; __any(open);) {
                if (!open) continue;
                U u = __hip_atomic_load(q, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                if (u == sent && spins++ < limit) continue;
                if (u == sent) {   // given up (the host reports it)
                    __hip_atomic_store(a.err, 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
                    u = Sentinel<TF>::nan;
                }
                __hip_atomic_store(cell(8u * (kBandRows + h)), u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                open = false;
            }
        }
    } else {
        // One wave issues an instruction every four cycles, so a slice costs about as many cycles as four
        // times its instructions, plus one LDS round trip: hence whole planes, byte offsets, and one test
        // for everything unusual (a value of another band that is not there yet reads as a NaN too).
        using P = SlicePlanes<W, TS>;
        const int ns = a.soff[band + 1] - a.soff[band];   // a multiple of 8
        const char* p = a.data + (size_t)a.soff[band] * P::bytes;
        BandSlot<W, TS> ring[D];
#pragma unroll
        for (int u = 0; u < D; ++u) band_load<W, TS, UNIT>(ring[u], p + (size_t)u * P::bytes, lane);
        auto lds = [&](unsigned at) {
            return __hip_atomic_load(cell(at), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
        };
        for (int s = 0; s < ns; s += D) {
            p += (size_t)D * P::bytes;
#pragma unroll
            for (int u = 0; u < D; ++u) {
                BandSlot<W, TS>& t = ring[u];
                const TF own = __builtin_bit_cast(TF, lds(t.row));
                U yv[W];
#pragma unroll
                for (int k = 0; k < W; ++k) yv[k] = lds(t.at[k]);
                TF r = own;
#pragma unroll
                for (int k = 0; k < W; ++k) r -= (TF)t.v[k] * __builtin_bit_cast(TF, yv[k]);
                if constexpr (!UNIT) r = quotient(r, (TF)t.d, t.ri);
                bool odd = UNIT ? r != r : !quotient_ok(r);
                if (__any(odd)) {
                    // wait for the halo (the other waves put a value there in the end), then the plain form
                    bool wait;
                    do {
                        wait = false;
#pragma unroll
                        for (int k = 0; k < W; ++k) {
                            yv[k] = lds(t.at[k]);
                            wait |= yv[k] == sent;
                        }
                    } while (__any(wait));
                    if (odd) {
                        r = own;
#pragma unroll
                        for (int k = 0; k < W; ++k) r -= (TF)t.v[k] * __builtin_bit_cast(TF, yv[k]);
                        if constexpr (!UNIT) r = r / (TF)t.d;
                    }
                }
                __hip_atomic_store(cell(t.row), __builtin_bit_cast(U, r), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                // the wave's LDS accesses stay in this order: lanes read what other lanes of the wave wrote, and
                // the publishing wave finds a slice's values once it sees it counted
                __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
                __hip_atomic_store(&solved, s + u + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_WORKGROUP);
                band_load<W, TS, UNIT>(t, p + (size_t)u * P::bytes, lane);
            }
        }
    }
    __syncthreads();
    if constexpr (!UPPER) {
        // the backward sweep's input (the published rows once more, the same values)
        for (int i = tid; i < cnt; i += kBlock) {
            U u = *cell(8u * i);
            if (u == sent) u = Sentinel<TF>::nan;
            reinterpret_cast<U*>(a.sy)[r0 + i] = u;
        }
    } else {
        double v[1] = {0.0};
        for (int i = tid; i < cnt; i += kBlock) {
            const TV z = (TV)y[i].v;
            if (a.part) v[0] += (double)(a.src[r0 + i] * z);
            if ((const void*)a.out != (const void*)a.sw) a.out[r0 + i] = z;
        }
        if (a.part) block_partials<1>(v, a.part, band);
    }
}

// The slices with new factor values f, one lane per slot
template <typename TS, int W>
__global__ void k_band_fill(int slots, const int* __restrict__ pos, const int* __restrict__ grow,
                            const unsigned short* __restrict__ place, const int* __restrict__ diag,
                            const TS* __restrict__ f, char* __restrict__ data)
{
    using P = SlicePlanes<W, TS>;
    const int s = blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= slots) return;
    char* p = data + (size_t)(s >> 6) * P::bytes;
    const int lane = s & 63;
    constexpr int per = 16 / (int)sizeof(TS);
    for (int k = 0; k < W; ++k) {
        const int q = pos[(size_t)s * W + k];
        reinterpret_cast<TS*>(p + 1024 * (k / per) + 16 * lane)[k % per] = q >= 0 ? f[q] : (TS)0;
        reinterpret_cast<unsigned*>(p + P::place + 1024 * (k / 4) + 16 * lane)[k % 4] =
            8u * place[(size_t)s * (W + 1) + k];
    }
    reinterpret_cast<unsigned*>(p + P::row)[lane] = 8u * place[(size_t)s * (W + 1) + W];
    const double d = grow[s] >= 0 ? (double)f[diag[grow[s]]] : 1.0;
    double* o = reinterpret_cast<double*>(p + P::diag + 16 * lane);
    o[0] = d;
    o[1] = fabs(d) >= 0x1p-100 && fabs(d) <= 0x1p100 ? 1.0 / d : __builtin_nan("");
}

// ---- host side
// One triangle (part 0 strictly lower, 1 strictly upper); false if a band's halo or a row does not fit.
static bool build_triangle(Context* c, const Pattern& F, const std::vector<int>& lev, int part, int rows, int bands,
                           BandTriangle& T, int& slices, int& max_halo)
{
    const int n = F.n;
    auto k0 = [&](int i) { return part == 1 ? F.h_diag[i] + 1 : F.h_rowptr[i]; };
    auto k1 = [&](int i) { return part == 0 ? F.h_diag[i] : F.h_rowptr[i + 1]; };
    int width = 0;
    for (int i = 0; i < n; ++i) width = std::max(width, k1(i) - k0(i));
    if (width > 16) return false;
    const int W = T.width = width <= 4 ? 4 : width <= 8 ? 8 : 16;
    std::vector<int> soff(1, 0), hoff(1, 0), halo, pos, grow;
    std::vector<unsigned short> at_all;
    std::vector<int> place(n, -1), order, slice_of(n);
    slices = max_halo = 0;
    const unsigned short zero = kBandRows + kBandHalo, idle = zero + 1;
    auto pad = [&](int slots) {
        pos.resize((size_t)slots * W, -1);
        for (size_t q = grow.size(); q < (size_t)slots; ++q) {
            at_all.insert(at_all.end(), W, zero);
            at_all.push_back(idle);
        }
        grow.resize(slots, -1);
    };
    for (int b = 0; b < bands; ++b) {
        const int r0 = b * rows, r1 = std::min(n, r0 + rows);
        order.resize(r1 - r0);
        for (int i = r0; i < r1; ++i) order[i - r0] = i;
        std::stable_sort(order.begin(), order.end(), [&](int u, int v) { return lev[u] < lev[v]; });
        int slot = 64 * soff[b];
        for (size_t o = 0; o < order.size(); ++o) {
            if (o > 0 && lev[order[o]] != lev[order[o - 1]]) slot = (slot + 63) / 64 * 64;
            pad(slot + 1);
            const int i = order[o];
            grow[slot] = i;
            slice_of[i] = slot / 64 - soff[b];
            at_all[(size_t)slot * (W + 1) + W] = (unsigned short)(i - r0);
            for (int k = k0(i); k < k1(i); ++k) {
                const int j = F.h_col[k];
                int at = j - r0;
                if (j < r0 || j >= r1) {
                    if (place[j] < hoff[b]) {
                        place[j] = (int)halo.size();
                        halo.push_back(j);
                    }
                    at = kBandRows + place[j] - hoff[b];
                    if (place[j] - hoff[b] >= kBandHalo) return false;
                }
                pos[(size_t)slot * W + (k - k0(i))] = k;
                at_all[(size_t)slot * (W + 1) + (k - k0(i))] = (unsigned short)at;
            }
            ++slot;
        }
        const int used = (slot + 63) / 64 - soff[b];
        slices = std::max(slices, used);
        soff.push_back(soff[b] + (used + 7) / 8 * 8);
        pad(64 * soff[b + 1]);
        hoff.push_back((int)halo.size());
        max_halo = std::max(max_halo, hoff[b + 1] - hoff[b]);
    }
    pad(64 * (soff[bands] + 8));   // the last band's loads run ahead
    // the rows other bands wait for, by the slice that solves them
    std::vector<int> ooff(1, 0), out_at, mine;
    std::vector<char> wanted(n, 0);
    for (int j : halo) wanted[j] = 1;
    for (int b = 0; b < bands; ++b) {
        mine.clear();
        for (int i = b * rows; i < std::min(n, (b + 1) * rows); ++i)
            if (wanted[i]) mine.push_back(i);
        std::stable_sort(mine.begin(), mine.end(), [&](int u, int v) { return slice_of[u] < slice_of[v]; });
        for (int i : mine) out_at.insert(out_at.end(), {i - b * rows, slice_of[i]});
        ooff.push_back((int)out_at.size() / 2);
    }
    if (out_at.empty()) out_at.push_back(0);
    T.slices = soff[bands] + 8;
    if (halo.empty()) halo.push_back(0);
    upload(c, T.soff, soff);
    upload(c, T.hoff, hoff);
    upload(c, T.halo, halo);
    upload(c, T.ooff, ooff);
    upload(c, T.out_at, out_at);
    upload(c, T.pos, pos);
    upload(c, T.grow, grow);
    upload(c, T.place, at_all);
    return true;
}

std::unique_ptr<BandSweeps> band_build(Context* c, const Pattern& F, const std::vector<int>& lev,
                                       const std::vector<int>& ulev, int nlevels)
{
    auto b = std::make_unique<BandSweeps>();
    b->bands = (F.n + kBandRows - 1) / kBandRows;
    b->rows = (F.n + b->bands - 1) / b->bands;
    // A level of more rows than the bands have lanes takes several slices in turn in each of them: few large
    // levels (a random numbering: 18 levels at 65k rows) stay with the chunked sweeps, 103 us, which use the
    // whole chip for a level. The bound is the chunk size, where both have work for every workgroup.
    if (F.n / std::max(1, nlevels) > 256 * b->bands) return nullptr;
    int sl = 0, su = 0, hl = 0, hu = 0;
    if (!build_triangle(c, F, lev, 0, b->rows, b->bands, b->lower, sl, hl)) return nullptr;
    if (!build_triangle(c, F, ulev, 1, b->rows, b->bands, b->upper, su, hu)) return nullptr;
    b->max_halo = std::max(hl, hu);
    PFEM_HIP(hipStreamSynchronize(c->stream));
    return b;
}

template <typename TS, int W>
static void fill(Context* c, const BandTriangle& t, const Pattern& F, const TS* f, DevArray<char>& data)
{
    const int slots = 64 * t.slices;
    if (!data.p) data.alloc((size_t)t.slices * SlicePlanes<W, TS>::bytes);
    hipLaunchKernelGGL((k_band_fill<TS, W>), dim3(blocks_for(slots)), dim3(kBlock), 0, c->stream, slots, t.pos.p, t.grow.p,
                       t.place.p, F.diag.p, f, data.p);
}

template <typename TS>
static void fill(Context* c, const BandTriangle& t, const Pattern& F, const TS* f, DevArray<char>& data)
{
    if (t.width == 4) fill<TS, 4>(c, t, F, f, data);
    else if (t.width == 8) fill<TS, 8>(c, t, F, f, data);
    else fill<TS, 16>(c, t, F, f, data);
}

void band_refresh(Context* c, BandSweeps& b, const Pattern& F, const double* fac, const float* fac32)
{
    for (BandTriangle* t : {&b.lower, &b.upper}) {
        fill<double>(c, *t, F, fac, t->data);
        if (fac32) fill<float>(c, *t, F, fac32, t->data32);
    }
}

template <typename TV, typename TS, typename TF, bool UPPER, bool UNIT>
static void launch_triangle(Context* c, int bands, const BandTriangle& t, BandArgs<TV, TS, TF> a)
{
    a.soff = t.soff.p;
    a.hoff = t.hoff.p;
    a.halo = t.halo.p;
    a.ooff = t.ooff.p;
    a.out_at = t.out_at.p;
    a.data = sizeof(TS) == 8 ? t.data.p : t.data32.p;
    const dim3 g(bands), bl(kBlock);
    if (t.width == 4) hipLaunchKernelGGL((k_band_sweep<TV, TS, TF, 4, UPPER, UNIT>), g, bl, 0, c->stream, a);
    else if (t.width == 8) hipLaunchKernelGGL((k_band_sweep<TV, TS, TF, 8, UPPER, UNIT>), g, bl, 0, c->stream, a);
    else hipLaunchKernelGGL((k_band_sweep<TV, TS, TF, 16, UPPER, UNIT>), g, bl, 0, c->stream, a);
}

template <typename TV, typename TS, typename TF>
int band_sweeps(Context* c, const BandSweeps& b, int n, bool unit, const TV* src, TV* out, TF* sy, TF* sw, double* part,
                const int* done, int* err, int limit)
{
    BandArgs<TV, TS, TF> a{};
    a.n = n;
    a.rows = b.rows;
    a.src = src;
    a.out = out;
    a.sy = sy;
    a.sw = sw;
    a.part = part;
    a.done = done;
    a.err = err;
    a.limit = limit;
    if (unit) launch_triangle<TV, TS, TF, false, true>(c, b.bands, b.lower, a);
    else launch_triangle<TV, TS, TF, false, false>(c, b.bands, b.lower, a);
    launch_triangle<TV, TS, TF, true, false>(c, b.bands, b.upper, a);
    return b.bands;
}

template int band_sweeps<double, double, double>(Context*, const BandSweeps&, int, bool, const double*, double*, double*,
                                                 double*, double*, const int*, int*, int);
template int band_sweeps<double, float, double>(Context*, const BandSweeps&, int, bool, const double*, double*, double*,
                                                double*, double*, const int*, int*, int);
template int band_sweeps<float, float, float>(Context*, const BandSweeps&, int, bool, const float*, float*, float*, float*,
                                              double*, const int*, int*, int);

}  // namespace pfem
