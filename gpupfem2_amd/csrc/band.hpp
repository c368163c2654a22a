// Band sweeps (band.hip): triangular solves of a factor with many small dependency levels.
#pragma once

#include "internal.hpp"

namespace pfem {

// One triangle by bands of consecutive rows. A band's rows are listed in slices of up to 64 rows of one level,
// levels ascending, one row to a lane. A slice is one block of memory, in planes of 16 bytes a lane (an
// instruction's load is then 1 KB of consecutive bytes): W values, {diagonal, its reciprocal}, W places of the
// entries' values in the band's LDS, and a plane of 4 bytes a lane with the place of the row's own value
// (places as byte offsets).
struct BandTriangle {
    int width = 0;                  // W: 4, 8 or 16 entries a row
    long slots = 0;                 // lanes of all slices, padding included
    DevArray<int> soff, hoff;       // slice and halo ranges of each band (bands + 1)
    DevArray<int> halo;             // columns of other bands, in the order of their first use
    DevArray<int> ooff, out_at;     // {place, slice} of the rows other bands use, and each band's range of them
    DevArray<int> row;              // row of each slot (-1 unused)
    DevArray<char> data, data32;    // the slices with the FP64 factor and with its FP32 copy
};

struct BandSweeps {
    int rows = 0, bands = 0;
    BandTriangle lower, upper;
    DevArray<unsigned short> place; // of every factor entry's value in its band's LDS
};

// The plan of a factor pattern with its forward and backward levels, or null where the chunked sweeps are
// the better form (large levels, a halo that does not fit, slices that take too much memory).
std::unique_ptr<BandSweeps> band_build(Context* c, const Pattern& F, const std::vector<int>& lev,
                                       const std::vector<int>& ulev, int nlevels);
// New factor values (fac32 may be null); false if the FP32 slices would take too much memory
bool band_refresh(Context* c, BandSweeps& b, const Pattern& F, const double* fac, const float* fac32);
// out = U^-1 L^-1 src (unit: L has a unit diagonal) through the published buffers sy and sw; part (or null)
// receives the partials of (src, out), one per band. Returns the bands.
template <typename TV, typename TS, typename TF>
int band_sweeps(Context* c, const BandSweeps& b, int n, bool unit, const TV* src, TV* out, TF* sy, TF* sw, double* part,
                const int* done, int* err, int limit);

}  // namespace pfem
