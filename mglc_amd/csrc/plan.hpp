// plan.hpp -- which kernels make a context's steps.  Internal to
// libmglc_lbm.so.
#pragma once
#include "block.hpp"
#include "pair.hpp"

// Several steps per launch: boxes with walls on all sides in the library's own
// launch shape (a caller's block shape, occupancy cap or transform names the
// one-step kernel).
struct StepPlan {
    enum Kind { ONE, PAIR, BLOCK } kind = ONE;
    lbm::PairTiles pair{};
    lbm::BlockTiles block{};
};

// The steps of one call as launches.  Launches of several steps come in even
// numbers: a call then ends in the lattice, the lid density and the force arrays
// that one launch per step would end in (an even call where it began), which a
// graph captured before or after it relies on.  group: steps of such a launch (1:
// none).
struct StepGroups {
    int ones, twos = 0, group;
    StepGroups(int nsteps, int g) : ones(g == 1 ? nsteps : nsteps % (2 * g)), group(g) {
        if (g == 3 && ones >= 4) {  // of the up to five steps left two by two where that saves launches
            ones -= 4;
            twos = 2;
        }
    }
    int next() {
        if (ones > 0) return --ones, 1;
        if (twos > 0) return --twos, 2;
        return group;
    }
};

// The tiles of the buoyancy step's two-step kernel (thermal.hip).
bool thermal_pair_plan(const lbm_params& p, int cus, lbm::PairTiles* t);
