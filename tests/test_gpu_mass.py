"""What FP64 runs lose of the mass: MRT and buoyancy 2^-54 of it a step, the share
M^-1 in FP64 loses; BGK 2^-54 / tau, the share its FP64 weights (which sum to
1 - 2^-54) lose in omega (f - feq), as the oracle loses it too.  Bounds: 5 % of
that; what else rounding does to the mean of a few thousand cells is random and
thousands of times less."""
import math

import numpy as np
import pytest

from mglc_amd.lbm import Cavity, CavityConfig, ThermalConfig

pytestmark = pytest.mark.gpu

SHAPE, STEPS = (16, 14, 12), 6000


def change(rho):
    return math.fsum((rho - 1.0).ravel()) / rho.size


@pytest.mark.parametrize("kind,block_x", [("mrt", 0), ("mrt", 64), ("bgk", 0), ("bgk", 64), ("buoyancy", 0)])
def test_mass_lost(kind, block_x):
    print(f"[gpu] mass {kind} {block_x}", flush=True)
    tau = 0.58
    cfg = (ThermalConfig(*SHAPE, Rayleigh=1e4, N=16, block_x=block_x) if kind == "buoyancy"
           else CavityConfig(*SHAPE, tauf=tau, collision=kind, block_x=block_x, block_y=1 if block_x else 0))
    with Cavity(cfg) as c:
        c.initial()
        c.step(STEPS)
        got = change(c.macro()[0])
    share = STEPS * 2.0 ** -54 * (1.0 / tau if kind == "bgk" else 1.0)
    assert abs(got + share) <= 0.05 * share


def test_bgk_loses_what_the_oracle_loses(oracle_lib):
    O = oracle_lib
    tau = 0.58
    ref = O.cavity_run(O.cavity_params(*SHAPE, tau, 0.1, collision=O.BGK), STEPS, nthreads=0)[0]
    with Cavity(CavityConfig(*SHAPE, tauf=tau, collision="bgk")) as c:
        c.initial()
        c.step(STEPS)
        got = c.macro()[0]
    assert abs(change(np.asarray(got)) - change(np.asarray(ref))) <= 0.05 * STEPS * 2.0 ** -54 / tau
