// Resident PCG (resident.hip): plan and work space of a solver's single-launch solves.
#pragma once

#include "internal.hpp"

namespace pfem {

constexpr int kResTileNnz = 2048;   // kTileNnz of spmv.hpp: the non-zeros at which an SpMV tile ends

// A system's rows [row0, row0 + rows), its 256-row tiles [tile0, tile0 + ntiles) and its first workgroup
struct ResSys {
    int row0, rows, tile0, ntiles, blk0;
};

struct ResOut {
    double res;
    unsigned long long t0, tdone;   // device clock: start of the call, end of the system's solve
    int it, converged, nan, nrep;
};

struct ResidentWork {
    std::shared_ptr<Pattern> pat;
    std::vector<int> sys_rows, order;   // order[q]: the system at position q (largest first)
    int nsys = 0, blocks = 0, tiles = 0, largest = 0, width = 0;
    bool fits = false, tiles_permuted = false;
    int pause = 0;                      // solves to come that do not try: a wait has failed
    long given_up = 0;                  // solves in which one did
    DevArray<ResSys> sys;
    DevArray<double> ring, zbuf;
    DevArray<ResOut> out;
    DevArray<int> err;
    ResOut* h_out = nullptr;            // pinned: the results by position, then the error flag
    ~ResidentWork();

    // Systems [rows[k], rows[k + 1]) of a pattern; false if the launch-per-kernel path has to be taken.
    // single: one system whose sums follow the order of the pattern's SpMV tile table.
    bool plan(Context* c, std::shared_ptr<Pattern> p, const std::vector<int>& rows, bool single);
    // All systems in one launch; false (x as it was) if the grid does not fit the device,
    // a halo does not fit or a wait exceeded its limit. drop > 0: reliable updates. Results in h_out.
    template <typename T>
    bool solve(Context* c, const T* val, const T* invd, const T* b, T* x, bool x_zero, double tol, int tol_mode,
               int maxit, double drop, int spin_limit);
};

}  // namespace pfem
