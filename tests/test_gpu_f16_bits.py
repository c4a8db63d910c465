"""FP16-stored runs give the bits they always gave.  A store rounds by the last
bits of what is stored, so another order of the collision's operations sends a
run another way; the fixture (tests/golden/make_f16.py) holds fields from before
any kernel made several steps per launch."""
import os

import numpy as np
import pytest

from mglc_amd.lbm import Batch, Cavity, CavityConfig, ThermalConfig

pytestmark = pytest.mark.gpu

GOLDEN = os.path.join(os.path.dirname(__file__), "golden", "f16_bits.npz")
SHAPE = (12, 10, 9)
RUNS = {
    "mrt": dict(),
    "mrt_scale9": dict(f16_scale_log2=9),
    "mrt_meq12": dict(meq12_rho=1),
    "mrt_one_step": dict(block_x=64, block_y=1),
    "mrt_halo": dict(halo_faces=63, halo_loopback=1),
    "mrt_mfma_70x12x9": dict(transform="mfma"),
    "bgk": dict(collision="bgk"),
    "bgk_halo_y": dict(collision="bgk", halo_faces=12, halo_loopback=1),
    "thermal_x": dict(thermal_axis=0),
    "thermal_y_halo": dict(halo_faces=3, halo_loopback=1),
    "thermal_z_coriolis": dict(thermal_axis=2, Ekman=1e-3),
    "batch_mrt": dict(collision="mrt"),
    "batch_bgk": dict(collision="bgk"),
}


def run(name):
    kw = RUNS[name]
    nx, ny, nz = shape = (70, 12, 9) if name.endswith("70x12x9") else SHAPE
    rng = np.random.default_rng(3)
    start = [np.ones((nz, ny, nx))] + [rng.uniform(-0.02, 0.02, (nz, ny, nx)) for _ in range(3)]
    if name.startswith("batch"):
        cfgs = [CavityConfig(*s, tauf=0.58, U0=0.05 + 0.01 * m, storage="f16", **kw)
                for m, s in enumerate([(5, 4, 6), (17, 6, 5)])]
        with Batch(cfgs) as b:
            b.initial()
            b.step(107)
            return np.concatenate([x.ravel() for m in range(len(cfgs)) for x in b.macro(m)])
    thermal = name.startswith("thermal")
    cfg = (ThermalConfig(*shape, Rayleigh=2e4, N=12, storage="f16", **kw) if thermal
           else CavityConfig(*shape, tauf=0.58, U0=0.1, storage="f16", **kw))
    with Cavity(cfg) as c:
        c.load_fields(*start, *([rng.uniform(-0.4, 0.4, (nz, ny, nx))] if thermal else []))
        c.step(31)
        c.step(6)
        out = [*c.macro()] + ([c.temperature()] if thermal else [])
    return np.concatenate([x.ravel() for x in out])


@pytest.mark.parametrize("name", RUNS)
def test_fields_are_the_fixtures_bits(name):
    print(f"[gpu] f16 bits {name}", flush=True)
    assert np.array_equal(run(name), np.load(GOLDEN)[name])
