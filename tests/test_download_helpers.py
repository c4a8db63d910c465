"""CPU test of the staged downloads' helper threads (tests/download_helpers_check.c):
a download does not wait for helpers that get no CPU, they find nothing to do when
they start, the last context waits for them, and with or without them every byte
arrives."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(not shutil.which("gcc"), reason="gcc not available")
def test_helpers_are_not_waited_for(tmp_path, hip_lib):
    exe, lib = tmp_path / "check", os.path.join(ROOT, "mglc_amd")
    subprocess.run(["gcc", "-O1", "-rdynamic", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(ROOT, "tests", "download_helpers_check.c"), "-o", str(exe),
                    f"-L{lib}", "-lmglc_lbm", f"-Wl,-rpath,{lib}", "-Wl,--allow-shlib-undefined", "-lpthread", "-ldl"],
                   check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stdout + r.stderr
