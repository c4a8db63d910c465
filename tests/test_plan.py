"""CPU test of which boxes are stepped several steps per launch (on a device of 256
CUs): those measured slower that way than one step per launch, rows of 13 to 32
cells in a cached box above all, are not; those measured faster are.  Against
stand-ins for the runtime's memory calls, in a process of their own."""
import shutil
import subprocess
import sys

import pytest

from test_step_memory import ROOT, build_shim

PROGRAM = """
import ctypes, sys
ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
sys.path.insert(0, sys.argv[2])
from mglc_amd.lbm import Cavity, CavityConfig, ThermalConfig

def steps(kind, box, storage, loop=0, ekman=None):
    cfg = (CavityConfig(*box, tauf=0.6, storage=storage, halo_loopback=loop) if kind == "flow"
           else ThermalConfig(*box, Rayleigh=2e4, N=max(box), storage=storage, Ekman=ekman))
    with Cavity(cfg) as c:
        return c.plan()[0]

# measured in pairs (blocks for 83 x 15 x 25) at this share of the one-step kernel's speed
slower = [("flow", (14, 42, 154), "f32", 0, 0.83), ("flow", (16, 37, 149), "f32", 0, 0.85),
          ("flow", (13, 37, 161), "f32", 0, 0.87), ("flow", (29, 32, 56), "f64", 0, 0.87),
          ("flow", (15, 146, 46), "f32", 0, 0.89), ("flow", (13, 166, 50), "f32", 1, 0.92),
          ("flow", (27, 63, 31), "f64", 0, 0.96), ("flow", (83, 15, 25), "f32", 0, 0.96),
          ("buoyancy", (95, 66, 15), "f64", 0, 0.83), ("buoyancy", (50, 133, 15), "f64", 0, 0.84),
          ("buoyancy", (123, 56, 17), "f64", 0, 0.89), ("buoyancy", (64, 67, 26), "f64", 0, 0.92)]
faster = [("flow", (65, 65, 65), "f64", 0, 1.58), ("flow", (65, 65, 65), "f32", 0, 1.17),
          ("flow", (97, 66, 50), "f32", 0, 1.19), ("flow", (190, 97, 131), "f32", 0, 1.6),
          ("flow", (128, 128, 128), "f64", 1, 1.4), ("flow", (17, 17, 17), "f16", 0, 1.9),
          ("flow", (33, 33, 33), "f32", 0, 1.1), ("buoyancy", (51, 51, 51), "f64", 0, 1.2),
          ("buoyancy", (62, 55, 42), "f64", 0, 1.21), ("buoyancy", (128, 128, 128), "f32", 0, 1.5)]
wrong = [c for c in slower if steps(*c[:4]) != 1] + [c for c in faster if steps(*c[:4]) == 1]
assert not wrong, wrong
print("ok")
"""


@pytest.mark.skipif(not shutil.which("gcc"), reason="gcc not available")
def test_plans_follow_the_measurements(tmp_path):
    r = subprocess.run([sys.executable, "-c", PROGRAM, str(build_shim(tmp_path)), ROOT], capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
