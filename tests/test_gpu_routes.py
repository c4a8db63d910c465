"""Every kernel that makes several steps per launch, by the plan the library
reports (not by a guess from the box): bit for bit the one-step kernel, which a
caller's block shape selects, with blocks on every wall and, for the tiled ones,
blocks away from the x and y walls (three tiles or more each way); and the halo
that looped-back steps write for the next one, which walls on all sides never
read, against the packed state."""
import numpy as np
import pytest
import torch

from mglc_amd.lbm import NUM_REGIONS, Batch, Cavity, CavityConfig, ThermalConfig

pytestmark = pytest.mark.gpu

DTYPE = {"f64": torch.float64, "f32": torch.float32, "f16": torch.float16}


def start_fields(shape, seed=3):
    nx, ny, nz = shape
    rng = np.random.default_rng(seed)
    return [np.ones((nz, ny, nx))] + [rng.uniform(-0.02, 0.02, (nz, ny, nx)) for _ in range(3)]


# (kind of launch, box): blocks of cells with three and two steps, tiles walked along z
FLOW = [("block", 3, (17, 17, 17)), ("block", 2, (33, 33, 33)), ("tiles", 2, (256, 96, 64)), ("tiles", 2, (321, 79, 47))]


def halo_and_packed(c, storage):
    """The incoming halo and what the state sends out, per region (elements)."""
    n = c.halo_buffer_bytes() // {"f64": 8, "f32": 4, "f16": 2}[storage]
    got, sent = (torch.zeros(n, dtype=DTYPE[storage], device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    c.halo_incoming(got.data_ptr())
    c.halo_pack(sent.data_ptr())
    c.synchronize()
    got, sent = got.cpu().numpy(), sent.cpu().numpy()
    at = [c.halo_layout(r) for r in range(NUM_REGIONS)]
    return [got[o:o + k] for o, k in at], [sent[o:o + k] for o, k in at]


# (FP16 has no tiled kernel)
FLOW_RUNS = [(*f, st) for f in FLOW for st in ("f64", "f32", "f16") if f[0] == "block" or st != "f16"]


@pytest.mark.parametrize("collision", ["mrt", "bgk"])
@pytest.mark.parametrize("loop", [0, 1])
@pytest.mark.parametrize("kind,steps,shape,storage", FLOW_RUNS,
                         ids=[f"{k}{n}_{'x'.join(map(str, b))}_{st}" for k, n, b, st in FLOW_RUNS])
def test_flow(kind, steps, shape, storage, loop, collision):
    print(f"[gpu] route {kind} {shape} {storage} {collision} loop={loop}", flush=True)
    start = start_fields(shape)
    kw = dict(tauf=0.58, U0=0.1, storage=storage, collision=collision, halo_loopback=loop)
    with Cavity(CavityConfig(*shape, **kw)) as a, Cavity(CavityConfig(*shape, block_x=64, block_y=1, **kw)) as b:
        per_launch, blocks = a.plan()
        assert per_launch == steps and b.plan() == (1, (0, 0, 0))
        assert kind == "block" or min(blocks[:2]) >= 3
        for c in (a, b):
            c.load_fields(*start)
        for n in (2 * steps, 1, 2 * steps + 1, 4 * steps, 5):
            for c in (a, b):
                c.step(n)
            for x, y, name in zip(a.macro(), b.macro(), ("rho", "u", "v", "w")):
                assert np.array_equal(x, y), (n, name, float(np.abs(x - y).max()))
            assert a.check() == b.check()
            if loop:
                got, sent = halo_and_packed(a, storage)
                for r in range(NUM_REGIONS):
                    assert np.array_equal(got[r], sent[r ^ 1 if r < 6 else r]), (n, r)


# storage, axis of the held walls, Ekman number, box
BUOYANCY = [("f64", 1, None, (128, 40, 36)), ("f64", 2, 1e-3, (192, 100, 64)), ("f32", 0, None, (256, 64, 64)),
            ("f32", 1, 1e-3, (300, 70, 90)), ("f32", 2, None, (128, 128, 128))]


@pytest.mark.parametrize("storage,axis,ekman,shape", BUOYANCY)
def test_buoyancy(storage, axis, ekman, shape):
    nx, ny, nz = shape
    print(f"[gpu] route buoyancy {shape} {storage} {axis} {ekman}", flush=True)
    start = start_fields(shape) + [np.random.default_rng(5).uniform(-0.4, 0.4, (nz, ny, nx))]
    kw = dict(Rayleigh=2e4, N=max(shape), Ekman=ekman, thermal_axis=axis, storage=storage)
    with Cavity(ThermalConfig(*shape, **kw)) as a, Cavity(ThermalConfig(*shape, block_x=64, block_y=1, **kw)) as b:
        per_launch, blocks = a.plan()
        assert per_launch == 2 and b.plan()[0] == 1
        assert min(blocks[:2]) >= 3 or shape == (128, 128, 128)
        for c in (a, b):
            c.load_fields(*start)
        for n in (4, 7, 9):
            for c in (a, b):
                c.step(n)
            for x, y in zip((*a.macro(), a.temperature()), (*b.macro(), b.temperature())):
                assert np.array_equal(x, y), n
            assert a.check_thermal() == b.check_thermal() and a.nusselt() == b.nusselt()


@pytest.mark.parametrize("storage,collision", [("f64", "mrt"), ("f64", "bgk"), ("f32", "mrt"), ("f32", "bgk")])
def test_batch(storage, collision):
    shapes = [(n + d, n, n + 2 * d) for n in (33, 65, 48, 64, 64, 96) for d in (0, 3)] + [(160, 60, 20)]
    cfgs = [CavityConfig(*s, tauf=0.58, U0=0.05 + 0.003 * m, storage=storage, collision=collision)
            for m, s in enumerate(shapes)]
    print(f"[gpu] route batch {storage} {collision}", flush=True)
    with Batch(cfgs) as a, Batch(cfgs) as b:
        assert a.plan()[0] == 2
        for x in (a, b):
            x.initial()
        for n in (7, 2, 4, 106):
            a.step(n)
            b.step_each(n)
            for m in range(len(cfgs)):
                assert all(np.array_equal(x, y) for x, y in zip(a.macro(m), b.macro(m))), (n, shapes[m])
        a.set_launch(128, 300)
        assert a.plan()[:2] == (1, 300)


@pytest.mark.parametrize("pairs", [True, False])
def test_batch_keeps_its_graph(pairs):
    """Calls of an even number of steps replay the graph of the first one."""
    cfgs = [CavityConfig(n, n, n, tauf=0.58, storage="f32") for n in (64, 64, 48, 64, 65)]
    print(f"[gpu] route batch graphs {pairs}", flush=True)
    with Batch(cfgs) as b:
        if not pairs:
            b.set_launch(256, 300)
        assert b.plan()[0] == (2 if pairs else 1)
        b.initial()
        for n in (150, 102, 150, 4, 2, 198, 250):
            b.step(n)
        assert b.plan()[2] == 1
