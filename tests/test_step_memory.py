"""CPU tests of what launches of several steps keep beside the state: contexts and
batches that would not fit with it are made without, one step per launch, and
the second force array holds only the components in use.  Against stand-ins for
the runtime's memory calls (tests/hip_memory_shim.c), in a process of their own."""
import os
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
import ctypes, sys
shim = ctypes.CDLL(sys.argv[1], ctypes.RTLD_GLOBAL)
shim.shim_in_use.restype = ctypes.c_size_t
shim.shim_set_free.argtypes = [ctypes.c_size_t]
sys.path.insert(0, sys.argv[2])
from mglc_amd.lbm import Batch, Cavity, CavityConfig, ThermalConfig

def used(make):
    shim.shim_set_free(1 << 40)
    with make() as c:
        assert c.info().device_bytes <= shim.shim_in_use()
        got = c.plan()[0], shim.shim_in_use(), c.info().device_bytes
    assert shim.shim_in_use() == 0
    return got

kw = dict(Rayleigh=1e5, N=64)
for second, make, one in [
    # bytes of what two steps per launch need more: the lid density, the force, the lid densities and the tiles
    (8 * 64 * 64, lambda: Cavity(CavityConfig(64, 64, 64)), lambda: Cavity(CavityConfig(64, 64, 64, block_x=64, block_y=1))),
    ("force 3", lambda: Cavity(ThermalConfig(64, 64, 64, Ekman=1e-3, **kw)),
     lambda: Cavity(ThermalConfig(64, 64, 64, Ekman=1e-3, block_x=64, block_y=1, **kw))),
    ("force 1", lambda: Cavity(ThermalConfig(64, 64, 64, **kw)),
     lambda: Cavity(ThermalConfig(64, 64, 64, block_x=64, block_y=1, **kw))),
]:
    steps, most, counted = used(make)
    plain = used(one)
    assert steps == 2 and plain[0] == 1
    if isinstance(second, str):
        with make() as c:
            second = int(second[-1]) * 8 * c.info().pop_stride
    assert most - plain[1] == counted - plain[2] == second, (most - plain[1], second)
    for short in (1, second - 1, second):  # down to what one step per launch needs
        shim.shim_set_free(most - short)
        with make() as c:
            assert c.plan()[0] == 1 and shim.shim_in_use() == plain[1] and c.info().device_bytes == plain[2]
        assert shim.shim_in_use() == 0

cfgs = [CavityConfig(n, n, n, tauf=0.58, storage="f32") for n in (64, 64, 48, 64, 65)]
steps, most, counted = used(lambda: Batch(cfgs))
assert steps == 2
lid = 8 * sum(c.nx * c.ny for c in cfgs)
for short in (1, lid, lid + 24):
    shim.shim_set_free(most - short)
    with Batch(cfgs) as b:
        assert b.plan()[0] == 1
    assert shim.shim_in_use() == 0
print("ok")
"""


def build_shim(folder):
    shim = folder / "shim.so"
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "hip_memory_shim.c"), "-o", str(shim)], check=True)
    return shim


@pytest.mark.skipif(not shutil.which("gcc"), reason="gcc not available")
def test_without_room_for_several_steps(tmp_path):
    shim = build_shim(tmp_path)
    r = subprocess.run([sys.executable, "-c", PROGRAM, str(shim), ROOT], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
