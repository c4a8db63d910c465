"""CPU check that the halvings the wall-distance bisection takes at once
(calq_far_halvings of mglc_amd/csrc/sphere_geom.hpp) are exactly those of the
loop, for radii from below a node to the largest accepted, nodes just inside
the surface and grazing links included; and that most halvings are taken so."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not os.path.exists(HIPCC), reason="hipcc not available")
@pytest.mark.parametrize("lo,hi", [(0.05, 1.0), (1.0, 12.0), (100.0, 250.0)])
def test_halvings_taken_at_once_are_the_loops(tmp_path, lo, hi):
    exe = tmp_path / "calq_far_check"
    subprocess.run([HIPCC, "-x", "hip", "--cuda-host-only", "-O2", "-I", ROOT,
                    os.path.join(ROOT, "tests", "calq_far_check.hip"), "-o", str(exe)],
                   check=True, capture_output=True)
    out = subprocess.run([str(exe), str(lo), str(hi)], check=False, capture_output=True, text=True, timeout=120)
    print(out.stdout)
    fields = dict(zip(out.stdout.split()[0::2], map(int, out.stdout.split()[1::2])))
    assert out.returncode == 0 and fields["mismatches"] == 0
    assert fields["links"] > 300000 and fields["skipped"] > 10 * fields["links"]
