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
// correctly rounded quotient (quotient.hpp) at a third of the division's latency, so results are those of the
// sequential solve, bit for bit. A level takes 0.15 us in a chain, 0.2 us in a mesh (an apply's two solves of 399 levels: 160 us).
//
// Measured (MI355X, FP64 IC0 apply, chunked sweeps -> here): unit square 40k rows, 401 levels 1292 -> 147 us,
// 160k rows, 801 levels 4227 -> 321 us; cylinder 1M rows, 2689 levels 30.6 -> 1.64 ms; 3D box 133k rows, 151
// levels 1299 -> 187 us; tridiagonal, 8192 levels 13.2 -> 2.35 ms.
#include <algorithm>
#include <cmath>
#include <type_traits>

#include "band.hpp"
#include "device.hpp"
#include "quotient.hpp"
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

// Row i's entries of a triangle in the factor: strictly lower, or strictly upper
__device__ __forceinline__ int2 band_entries(bool upper, int i, const int* __restrict__ rowptr, const int* __restrict__ diag)
{
    return upper ? make_int2(diag[i] + 1, rowptr[i + 1]) : make_int2(rowptr[i], diag[i]);
}

constexpr unsigned kBandZero = kBandRows + kBandHalo, kBandIdle = kBandZero + 1;   // places of unused entries and lanes

// The planes of places, which only the pattern decides, one lane per slot
template <typename TS, int W>
__global__ void k_band_places(long slots, int rows, bool upper, const int* __restrict__ row, const int* __restrict__ rowptr,
                              const int* __restrict__ diag, const unsigned short* __restrict__ place,
                              char* __restrict__ data)
{
    using P = SlicePlanes<W, TS>;
    const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= slots) return;
    char* p = data + (size_t)(s >> 6) * P::bytes;
    const int lane = (int)(s & 63), i = row[s];
    const int2 e = i >= 0 ? band_entries(upper, i, rowptr, diag) : make_int2(0, 0);
    for (int k = 0; k < W; ++k)
        reinterpret_cast<unsigned*>(p + P::place + 1024 * (k / 4) + 16 * lane)[k % 4] =
            8u * (e.x + k < e.y ? place[e.x + k] : kBandZero);
    reinterpret_cast<unsigned*>(p + P::row)[lane] = 8u * (i >= 0 ? (unsigned)(i % rows) : kBandIdle);
}

// The other planes from the factor's values f
template <typename TS, int W>
__global__ void k_band_values(long slots, bool upper, const int* __restrict__ row, const int* __restrict__ rowptr,
                              const int* __restrict__ diag, const TS* __restrict__ f, char* __restrict__ data)
{
    using P = SlicePlanes<W, TS>;
    const long s = (long)blockIdx.x * blockDim.x + threadIdx.x;
    if (s >= slots) return;
    char* p = data + (size_t)(s >> 6) * P::bytes;
    const int lane = (int)(s & 63), i = row[s];
    constexpr int per = 16 / (int)sizeof(TS);
    const int2 e = i >= 0 ? band_entries(upper, i, rowptr, diag) : make_int2(0, 0);
    for (int k = 0; k < W; ++k)
        reinterpret_cast<TS*>(p + 1024 * (k / per) + 16 * lane)[k % per] = e.x + k < e.y ? f[e.x + k] : (TS)0;
    const double d = i >= 0 ? (double)f[diag[i]] : 1.0;
    double* o = reinterpret_cast<double*>(p + P::diag + 16 * lane);
    o[0] = d;
    o[1] = fabs(d) >= 0x1p-100 && fabs(d) <= 0x1p100 ? 1.0 / d : __builtin_nan("");
}

// f(W as a type) for the triangle's width
template <typename F>
static auto with_width(int width, F f)
{
    if (width == 4) return f(std::integral_constant<int, 4>());
    if (width == 8) return f(std::integral_constant<int, 8>());
    return f(std::integral_constant<int, 16>());
}

template <typename TS>
static size_t slice_bytes(int width)
{
    return with_width(width, [](auto w) { return (size_t)SlicePlanes<decltype(w)::value, TS>::bytes; });
}

// ---- host side
// One triangle (upper or lower) while it is planned
struct BandPlan {
    const Pattern& F;
    const std::vector<int>& lev;
    bool upper;
    int rows, bands, width = 0;
    std::vector<int> order;        // the rows of band b from b * rows on, by level, ascending within a level
    std::vector<int> soff;         // slices of each band
    double us = 0.0;               // of a solve, estimated
    int k0(int i) const { return upper ? F.h_diag[i] + 1 : F.h_rowptr[i]; }
    int k1(int i) const { return upper ? F.h_rowptr[i + 1] : F.h_diag[i]; }
    long slots() const { return 64L * (soff[bands] + 8); }   // the last band's loads run eight slices ahead

    // false if a row does not fit
    bool schedule()
    {
        const int n = F.n;
        for (int i = 0; i < n; ++i) width = std::max(width, k1(i) - k0(i));
        if (width > 16) return false;
        width = width <= 4 ? 4 : width <= 8 ? 8 : 16;
        std::vector<int> at(*std::max_element(lev.begin(), lev.end()) + 2, 0), by_level(n), next(bands);
        for (int l : lev) ++at[l + 1];
        for (size_t l = 1; l < at.size(); ++l) at[l] += at[l - 1];
        for (int i = 0; i < n; ++i) by_level[at[lev[i]]++] = i;
        order.resize(n);
        for (int b = 0; b < bands; ++b) next[b] = b * rows;
        for (int i : by_level) order[next[i / rows]++] = i;
        soff.assign(1, 0);
        for (int b = 0; b < bands; ++b) {
            long slot = 0;
            for (int o = b * rows; o < std::min(n, (b + 1) * rows); ++o, ++slot)
                if (o > b * rows && lev[order[o]] != lev[order[o - 1]]) slot = (slot + 63) / 64 * 64;
            soff.push_back(soff[b] + (int)((slot + 511) / 512 * 8));
        }
        return true;
    }

    // The time of a solve from that of a slice and of a value's way to another band; bands run ahead of each other as
    // far as their dependencies let them
    void estimate()
    {
        const double slice = width == 4 ? 0.144 : width == 8 ? 0.174 : 0.238, hop = 1.2;
        const int n = F.n;
        std::vector<double> solved(n);
        for (int q = 0; q < bands; ++q) {
            const int r0 = (upper ? bands - 1 - q : q) * rows, r1 = std::min(n, r0 + rows);
            double t = 0.0;
            for (int o = r0; o < r1;) {
                int end = o;   // of the slice
                while (end < r1 && end - o < 64 && lev[order[end]] == lev[order[o]]) ++end;
                for (int p = o; p < end; ++p)
                    for (int k = k0(order[p]); k < k1(order[p]); ++k)
                        if (const int j = F.h_col[k]; j < r0 || j >= r1) t = std::max(t, solved[j] + hop);
                t += slice;
                for (; o < end; ++o) solved[order[o]] = t;
            }
            us = std::max(us, t);
        }
    }

    // The triangle's tables; place: of every entry. False if a band's halo does not fit.
    bool build(Context* c, BandTriangle& T, std::vector<unsigned short>& place) const
    {
        const int n = F.n;
        std::vector<int> hoff(1, 0), halo, slot_row(slots(), -1), halo_at(n, -1), slice_of(n);
        for (int b = 0; b < bands; ++b) {
            const int r0 = b * rows, r1 = std::min(n, r0 + rows);
            long slot = 64L * soff[b];
            for (int o = r0; o < r1; ++o, ++slot) {
                const int i = order[o];
                if (o > r0 && lev[i] != lev[order[o - 1]]) slot = (slot + 63) / 64 * 64;
                slot_row[slot] = i;
                slice_of[i] = (int)(slot / 64) - soff[b];
                for (int k = k0(i); k < k1(i); ++k) {
                    const int j = F.h_col[k];
                    int at = j - r0;
                    if (j < r0 || j >= r1) {
                        if (halo_at[j] < hoff[b]) {
                            halo_at[j] = (int)halo.size();
                            halo.push_back(j);
                        }
                        if (halo_at[j] - hoff[b] >= kBandHalo) return false;
                        at = kBandRows + halo_at[j] - hoff[b];
                    }
                    place[k] = (unsigned short)at;
                }
            }
            hoff.push_back((int)halo.size());
        }
        // the rows other bands wait for, by the slice that solves them
        std::vector<int> ooff(1, 0), out_at, mine;
        std::vector<char> wanted(n, 0);
        for (int j : halo) wanted[j] = 1;
        for (int b = 0; b < bands; ++b) {
            for (int o = b * rows; o < std::min(n, (b + 1) * rows); ++o)
                if (wanted[order[o]]) out_at.insert(out_at.end(), {order[o] - b * rows, slice_of[order[o]]});
            ooff.push_back((int)out_at.size() / 2);
        }
        if (out_at.empty()) out_at.push_back(0);
        if (halo.empty()) halo.push_back(0);
        T.width = width;
        T.slots = slots();
        upload(c, T.soff, soff);
        upload(c, T.hoff, hoff);
        upload(c, T.halo, halo);
        upload(c, T.ooff, ooff);
        upload(c, T.out_at, out_at);
        upload(c, T.row, slot_row);
        return true;
    }
};

template <typename TS>
static void lay_out(Context* c, const BandSweeps& b, const Pattern& F, bool upper, DevArray<char>& data)
{
    const BandTriangle& t = upper ? b.upper : b.lower;
    data.alloc((size_t)(t.slots / 64) * slice_bytes<TS>(t.width));
    with_width(t.width, [&](auto w) {
        hipLaunchKernelGGL((k_band_places<TS, decltype(w)::value>), dim3(blocks_for(t.slots)), dim3(kBlock), 0, c->stream,
                           t.slots, b.rows, upper, t.row.p, F.rowptr.p, F.diag.p, b.place.p, data.p);
    });
}

// A slice has 64 lanes however few rows of a level the band holds, so the slices grow with the levels times the
// bands: 0.6 KB a row and triangle for a mesh of 1000 lines, 4.6 KB for a chain. They may take a sixteenth of the
// device's memory (19 of 309 GB: meshes of 2500 lines, chains of 2M rows) and a quarter of what is free. Systems
// beyond take the chunked sweeps, whose tables are the factor's size.
static bool affordable(size_t bytes)
{
    size_t free = 0, total = 0;
    PFEM_HIP(hipMemGetInfo(&free, &total));
    return bytes <= std::min(total / 16, free / 4);
}

std::unique_ptr<BandSweeps> band_build(Context* c, const Pattern& F, const std::vector<int>& lev,
                                       const std::vector<int>& ulev, int nlevels)
{
    auto b = std::make_unique<BandSweeps>();
    b->bands = (F.n + kBandRows - 1) / kBandRows;
    b->rows = (F.n + b->bands - 1) / b->bands;
    BandPlan lower{F, lev, false, b->rows, b->bands}, upper{F, ulev, true, b->rows, b->bands};
    if (!lower.schedule() || !upper.schedule()) return nullptr;
    size_t bytes = 0;
    for (const BandPlan* p : {&lower, &upper}) bytes += (size_t)(p->slots() / 64) * (slice_bytes<double>(p->width) + 256);
    if (!affordable(bytes)) return nullptr;
    // The chunked sweeps use the whole chip for a level and take 1.06 to 1.6 us for a level of up to 7000 rows. A band
    // takes a level's rows 64 at a time, and bands whose levels do not overlap follow one another, so large levels
    // are slower here: us a solve in chunks and in bands (estimate), half bandwidths 2000 and 2001, 200k rows,
    // 100 levels: 136 and 640 (384); 1000, 60k rows, 60 levels: 64 and 173 (130); 300, 200 levels: 177 and 170 (148);
    // unit square of 40k rows, 401 levels: 650 and 80 (62); its numbering shuffled, 15 levels: 53 (62).
    lower.estimate();
    upper.estimate();
    if (lower.us + upper.us > 2.0 * nlevels) return nullptr;
    std::vector<unsigned short> place(F.nnz, 0);
    if (!lower.build(c, b->lower, place) || !upper.build(c, b->upper, place)) return nullptr;
    upload(c, b->place, place);
    lay_out<double>(c, *b, F, false, b->lower.data);
    lay_out<double>(c, *b, F, true, b->upper.data);
    PFEM_HIP(hipStreamSynchronize(c->stream));
    return b;
}

bool band_refresh(Context* c, BandSweeps& b, const Pattern& F, const double* fac, const float* fac32)
{
    if (fac32 && !b.lower.data32.p) {
        size_t bytes = 0;
        for (const BandTriangle* t : {&b.lower, &b.upper}) bytes += (size_t)(t->slots / 64) * slice_bytes<float>(t->width);
        if (!affordable(bytes)) return false;
        lay_out<float>(c, b, F, false, b.lower.data32);
        lay_out<float>(c, b, F, true, b.upper.data32);
    }
    for (bool upper : {false, true}) {
        BandTriangle& t = upper ? b.upper : b.lower;
        with_width(t.width, [&](auto w) {
            constexpr int W = decltype(w)::value;
            const dim3 g(blocks_for(t.slots)), bl(kBlock);
            hipLaunchKernelGGL((k_band_values<double, W>), g, bl, 0, c->stream, t.slots, upper, t.row.p, F.rowptr.p,
                               F.diag.p, fac, t.data.p);
            if (fac32)
                hipLaunchKernelGGL((k_band_values<float, W>), g, bl, 0, c->stream, t.slots, upper, t.row.p, F.rowptr.p,
                                   F.diag.p, fac32, t.data32.p);
        });
    }
    return true;
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
    with_width(t.width, [&](auto w) {
        hipLaunchKernelGGL((k_band_sweep<TV, TS, TF, decltype(w)::value, UPPER, UNIT>), dim3(bands), dim3(kBlock), 0,
                           c->stream, a);
    });
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
