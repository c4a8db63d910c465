"""Fields come back from the device as they are there, whichever way the copy
takes (plain, or staged through pinned memory from 16 MiB on), at sizes that are
not whole staging slots, and for two contexts on two threads at once."""
import threading

import numpy as np
import pytest

from mglc_amd.lbm import Cavity, CavityConfig

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(64, 64, 60), (81, 80, 83), (130, 90, 75)], ids=lambda s: "x".join(map(str, s)))
def test_loaded_fields_come_back(shape):
    nx, ny, nz = shape
    rng = np.random.default_rng(11)
    fields = [[rng.uniform(0.9, 1.1, (nz, ny, nx)) for _ in range(4)] for _ in range(2)]
    print(f"[gpu] download {shape}", flush=True)
    with Cavity(CavityConfig(nx, ny, nz, tauf=0.6)) as a, Cavity(CavityConfig(nx, ny, nz, tauf=0.6)) as b:
        for c, f in zip((a, b), fields):
            c.load_fields(*f)
        bad = []

        def read(c, f):
            for _ in range(4):
                bad.extend(k for k, (x, y) in enumerate(zip(c.macro(), f)) if not np.array_equal(x, y))

        threads = [threading.Thread(target=read, args=p) for p in zip((a, b), fields)]
        for t in threads:
            t.start()
        for t in threads:
            t.join()
        assert not bad
