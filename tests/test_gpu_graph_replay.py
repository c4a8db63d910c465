"""A captured graph of steps goes on from wherever direct steps, replays or a new
start left the context: direct calls of several steps per launch end in the
buffers that one launch per step would end in.  Against a context that makes the
same steps one per launch (its own block shape), bit for bit."""
import ctypes

import numpy as np
import pytest

from mglc_amd.hip import Stream, runtime
from mglc_amd.lbm import Cavity, CavityConfig, ThermalConfig

pytestmark = pytest.mark.gpu

BOXES = {  # three steps per launch, two (blocks), two (tiles) with and without the looped-back halo, buoyancy
    "block3": ((17, 17, 17), CavityConfig, dict(tauf=0.58)),
    "block3_f32_loop": ((17, 17, 17), CavityConfig, dict(tauf=0.58, storage="f32", halo_loopback=1)),
    "block2": ((33, 33, 33), CavityConfig, dict(tauf=0.58)),
    "pair": ((65, 40, 70), CavityConfig, dict(tauf=0.58)),
    "pair_loop": ((128, 64, 64), CavityConfig, dict(tauf=0.58, halo_loopback=1)),
    "buoyancy": ((51, 51, 51), ThermalConfig, dict(Rayleigh=2e4, N=51)),
    "buoyancy_rot_f32": ((128, 128, 128), ThermalConfig, dict(Rayleigh=2e4, N=128, Ekman=1e-3, storage="f32")),
}


@pytest.mark.parametrize("name", BOXES)
def test_replays_between_direct_steps(name):
    shape, config, kw = BOXES[name]
    nx, ny, nz = shape
    rng = np.random.default_rng(3)
    starts = []
    for _ in range(2):
        s = [np.ones((nz, ny, nx))] + [rng.uniform(-0.02, 0.02, (nz, ny, nx)) for _ in range(3)]
        starts.append(s + ([rng.uniform(-0.4, 0.4, (nz, ny, nx))] if config is ThermalConfig else []))
    print(f"[gpu] graph replay {name}", flush=True)
    hip = runtime()
    stream, graph, ex = Stream(), ctypes.c_void_p(), ctypes.c_void_p()
    with Cavity(config(*shape, **kw), stream=stream.handle.value) as a, \
            Cavity(config(*shape, **kw, block_x=64, block_y=1), stream=stream.handle.value) as b:
        def same(what):
            fa, fb = ([*c.macro()] + ([c.temperature()] if config is ThermalConfig else []) for c in (a, b))
            assert all(np.array_equal(x, y) for x, y in zip(fa, fb)), what

        def both(n):
            a.step(n)
            b.step(n)
            same(f"{n} direct steps")

        def replay(what):
            assert hip.hipGraphLaunch(ex, stream.handle) == 0
            b.step(2)
            same(f"replay {what}")

        for c in (a, b):
            c.load_fields(*starts[0])
        both(2)  # before the capture, too
        assert hip.hipStreamBeginCapture(stream.handle, 2) == 0  # relaxed
        a.step(2)
        assert hip.hipStreamEndCapture(stream.handle, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
        try:
            replay("first")
            for n in (2, 4, 6, 8, 10, 12, 14):
                both(n)
                replay(f"after {n} direct steps")
            both(3)
            both(5)
            replay("after 3 and 5")
            for c in (a, b):
                c.load_fields(*starts[1])
            replay("from new fields")
            both(2)
            for c in (a, b):
                c.load_fields(*starts[0])
            replay("from the first fields")
        finally:
            hip.hipGraphExecDestroy(ex)
            hip.hipGraphDestroy(graph)
    stream.close()
