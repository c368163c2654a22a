// Resident IC0-PCG (resident_ic0.hip): plan and work space of a solver's single-launch solves.
#pragma once

#include "internal.hpp"
#include "solver.hpp"

namespace pfem {

struct ResidentIc0 {
    std::shared_ptr<Pattern> pat;   // the factor's pattern (factor ordering) that the plan is for
    std::vector<int> colours;       // row offsets of its colours
    bool fits = false;
    int blocks = 0, width = 0, places = 0;
    int pause = 0;                  // solves to come that do not try: a wait has failed
    long given_up = 0;              // solves in which one did
    DevArray<int> rows, halo, steps;   // per lane: row, halo row (or -1); per workgroup: sweep steps
    DevArray<int> post, from;          // per lane: exchange places of a row on a patch's rim, of a halo row
    DevArray<uint32_t> info, hinfo;
    DevArray<uint16_t> slot;                     // place of entry e of lane t at e * lanes + t
    DevArray<double> buf, ring;
    DevArray<CgState> out;
    DevArray<int> err;
    int* h_err = nullptr;           // pinned
    ~ResidentIc0();

    bool plan(Context* c, const pfem_precond_t* pc);
    // The iterations that follow the start of a PCG solve (r, p and st set); false (x, r, p, st as they were) if
    // the launch-per-kernel path has to take them. The state ends in hst.
    bool solve(Context* c, pfem_precond_t* pc, bool reduced, double* x, const double* r, const double* p,
               const CgState* st, CgState* hst);
};

}  // namespace pfem
