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

// The tiles of the buoyancy step's two-step kernel (thermal.hip).
bool thermal_pair_plan(const lbm_params& p, int cus, lbm::PairTiles* t);
