"""The kernels that make several steps per launch (pair.hpp: two steps, tiles
walked along z; block.hpp: two or three, one block of cells per workgroup)
against the one-step kernel, which a caller's block shape selects: every cell
makes the same operations, so fields, lid density and residual agree bit for
bit.  Shapes sit at the tiles' edges: one cell past a tile, boxes thinner than
a tile, one plane per chunk, odd numbers of steps (the rest goes one by one)."""
import ctypes

import numpy as np
import pytest

from mglc_amd.hip import Stream, runtime
from mglc_amd.lbm import Batch, Cavity, CavityConfig, ThermalConfig

pytestmark = pytest.mark.gpu

SHAPES = [(2, 2, 2), (3, 5, 4), (17, 17, 17), (24, 9, 31), (33, 30, 20),   # blocks, three and two steps
          (65, 65, 65), (33, 14, 200), (64, 40, 70), (97, 66, 50), (130, 27, 45), (66, 130, 30)]  # pairs


def run(shape, start, counts, **kw):
    nx, ny, nz = shape
    with Cavity(CavityConfig(nx, ny, nz, tauf=0.58, U0=0.1, **kw)) as c:
        c.load_fields(*start)
        errs = []
        for n in counts:
            c.step(n)
            errs.append(c.check())
        return c.macro(), errs


def start_fields(shape, seed=3):
    nx, ny, nz = shape
    rng = np.random.default_rng(seed)
    return [np.ones((nz, ny, nx))] + [rng.uniform(-0.02, 0.02, (nz, ny, nx)) for _ in range(3)]


@pytest.mark.parametrize("storage,collision,loop", [("f64", "mrt", 0), ("f64", "bgk", 1), ("f32", "mrt", 1),
                                                    ("f32", "bgk", 0), ("f16", "mrt", 0)])
@pytest.mark.parametrize("shape", SHAPES, ids=["x".join(map(str, s)) for s in SHAPES])
def test_several_steps_per_launch_equal_single_steps(shape, storage, collision, loop):
    start = start_fields(shape)
    kw = dict(storage=storage, collision=collision, halo_loopback=loop)
    print(f"[gpu] multistep {shape} {kw}", flush=True)
    got, errs = run(shape, start, (7, 1, 6), **kw)
    ref, errs1 = run(shape, start, (7, 1, 6), block_x=64, block_y=1, **kw)
    for g, r, name in zip(got, ref, ("rho", "u", "v", "w")):
        assert np.array_equal(g, r), (name, float(np.abs(g - r).max()))
    assert errs == errs1


def test_restart_between_groups_of_steps():
    """A state saved after an odd number of steps goes on in another context."""
    shape = (65, 40, 70)
    start = start_fields(shape)
    with Cavity(CavityConfig(*shape, tauf=0.58)) as a, Cavity(CavityConfig(*shape, tauf=0.58)) as b:
        a.load_fields(*start)
        a.step(5)
        b.load_state(a.save_state())
        a.step(9)
        b.step(4)
        b.step(5)
        for g, r in zip(a.macro(), b.macro()):
            assert np.array_equal(g, r)


THERMAL_SHAPES = [(3, 4, 5), (33, 30, 40), (51, 51, 51), (64, 31, 90), (128, 40, 36), (65, 100, 33)]


@pytest.mark.parametrize("storage,axis,ekman", [("f64", 1, None), ("f64", 2, 1e-3), ("f32", 0, None),
                                                ("f32", 1, 1e-3)])
@pytest.mark.parametrize("shape", THERMAL_SHAPES, ids=["x".join(map(str, s)) for s in THERMAL_SHAPES])
def test_two_buoyancy_steps_per_launch_equal_single_steps(shape, storage, axis, ekman):
    nx, ny, nz = shape
    start = start_fields(shape)
    T = np.random.default_rng(5).uniform(-0.4, 0.4, (nz, ny, nx))
    print(f"[gpu] multistep thermal {shape} {storage} {axis} {ekman}", flush=True)
    out = []
    for kw in (dict(), dict(block_x=64, block_y=1)):
        cfg = ThermalConfig(nx, ny, nz, Rayleigh=2e4, N=max(shape), Ekman=ekman, thermal_axis=axis, storage=storage, **kw)
        with Cavity(cfg) as c:
            c.load_fields(*start, T)
            c.step(7)
            e1 = c.check_thermal()
            c.step(6)
            out.append((*c.macro(), c.temperature(), np.array([e1, c.check_thermal(), c.nusselt()])))
    for g, r, name in zip(*out, ("rho", "u", "v", "w", "T", "sums")):
        assert np.array_equal(g, r), (name, float(np.abs(g - r).max()))


def test_steps_captured_into_a_graph_replay():
    """Under stream capture steps go one per launch, so a graph of an even number
    of them leaves the buffers in place and every replay goes on from the last."""
    shape = (65, 40, 70)
    start = start_fields(shape)
    hip = runtime()
    stream, graph, ex = Stream(), ctypes.c_void_p(), ctypes.c_void_p()
    with Cavity(CavityConfig(*shape, tauf=0.58), stream=stream.handle.value) as a, \
            Cavity(CavityConfig(*shape, tauf=0.58), stream=stream.handle.value) as b:
        for c in (a, b):
            c.load_fields(*start)
            c.step(2)
            c.synchronize()
        assert hip.hipStreamBeginCapture(stream.handle, 2) == 0  # relaxed
        a.step(4)
        assert hip.hipStreamEndCapture(stream.handle, ctypes.byref(graph)) == 0
        assert hip.hipGraphInstantiate(ctypes.byref(ex), graph, None, None, ctypes.c_size_t(0)) == 0
        try:
            for _ in range(3):
                assert hip.hipGraphLaunch(ex, stream.handle) == 0
                b.step(4)
                for x, y in zip(a.macro(), b.macro()):
                    assert np.array_equal(x, y)
        finally:
            hip.hipGraphExecDestroy(ex)
            hip.hipGraphDestroy(graph)
    stream.close()


@pytest.mark.parametrize("storage,collision", [("f64", "mrt"), ("f64", "bgk"), ("f32", "mrt"), ("f32", "bgk")])
def test_batch_of_two_steps_per_launch_equals_one_launch_per_instance(storage, collision):
    """Uneven boxes (one plane per chunk up to several tiles each way), odd step
    counts, a graph replay, and one-step launches in between."""
    shapes = [(n + d, n, n + 2 * d) for n in (5, 17, 33, 65, 48, 64, 64, 64) for d in (0, 3)]
    cfgs = [CavityConfig(*s, tauf=0.58, U0=0.05 + 0.005 * m, storage=storage, collision=collision)
            for m, s in enumerate(shapes)]
    print(f"[gpu] multistep batch {storage} {collision}", flush=True)
    with Batch(cfgs) as a, Batch(cfgs) as b:
        a.initial()
        b.initial()
        for n in (7, 2, 201):
            a.step(n)
            b.step_each(n)
            for m in range(len(cfgs)):
                assert all(np.array_equal(x, y) for x, y in zip(a.macro(m), b.macro(m))), (n, shapes[m])
        a.set_launch(128, 300)
        a.step(103)
        b.step_each(103)
        for m in range(len(cfgs)):
            assert all(np.array_equal(x, y) for x, y in zip(a.macro(m), b.macro(m))), shapes[m]
