"""The second force array that launches of two buoyancy steps keep beside the state
never gets into a saved state."""
import numpy as np
import pytest

from mglc_amd.lbm import Cavity, ThermalConfig

pytestmark = pytest.mark.gpu


def written(blob, shape, stride):
    """The state's arrays (all FP64 here) without what no kernel writes: between a
    population's last cell and the next population, and a lid density, which a
    buoyancy context has no lid for."""
    nx, ny, nz = shape
    n = nx * ny * nz
    counts = [19 * stride, nx * ny, 4 * n, 2 * n, 7 * stride, 3 * stride, n, 2 * n]  # f, lid, fields, g, force, T
    data = np.frombuffer(blob, dtype=np.uint64, offset=len(blob) - 8 * sum(counts))
    parts = np.split(data, np.cumsum(counts)[:-1])
    return np.concatenate([x.reshape(-1, stride)[:, :n].ravel() if k in (0, 4, 5) else x
                           for k, x in enumerate(parts) if k != 1])


def test_saved_state_is_the_one_step_runs():
    shape = (128, 40, 36)  # rows without padding
    rng = np.random.default_rng(3)
    start = [np.ones(shape[::-1])] + [rng.uniform(-0.02, 0.02, shape[::-1]) for _ in range(3)]
    start.append(rng.uniform(-0.4, 0.4, shape[::-1]))
    kw = dict(Rayleigh=2e4, N=128)
    print("[gpu] step memory state", flush=True)
    with Cavity(ThermalConfig(*shape, **kw)) as a, Cavity(ThermalConfig(*shape, block_x=64, block_y=1, **kw)) as b, \
            Cavity(ThermalConfig(*shape, Ekman=1e-3, **kw)) as rot, \
            Cavity(ThermalConfig(*shape, Ekman=1e-3, block_x=64, block_y=1, **kw)) as rot_one:
        assert a.plan()[0] == 2 and rot.plan()[0] == 2
        for c in (a, b):
            c.load_fields(*start)
        for n in (2, 4, 5):
            for c in (a, b):
                c.step(n)
                c.check_thermal()
            stride = a.info().pop_stride
            x, y = (written(c.save_state(), shape, stride) for c in (a, b))
            assert np.array_equal(x, y), n
        for c, source in ((rot, a), (rot_one, b)):  # takes Fx and Fy of the state as the last collision's
            c.load_state(source.save_state())
            c.step(4)
        for x, y in zip((*rot.macro(), rot.temperature()), (*rot_one.macro(), rot_one.temperature())):
            assert np.array_equal(x, y)
