"""Worlds that several workgroups colour and sweep, against the same worlds
with one workgroup each and against the oracle's restatement: every bit."""
import numpy as np
import pytest

from shapes_amd import engine, scenes
from test_gpu_colored import _colored_vs_restatement

pytestmark = pytest.mark.gpu

MIN_BODIES, GROUP_BODIES, GROUP_MAX, MAX_GROUPS = 2048, 64, 384, 256


def _world(n, seed=78, cols=200):
    rng = np.random.Generator(np.random.Philox(seed))
    return scenes.grid_world(rng, n, cols=cols, spacing=1.05, y0=1.0, square_frac=0.5, vel=0.3)


def _shared(worlds, cfg, **kw):
    """Workgroups of the sweeps beyond one to a world."""
    st, msg, p, rows = engine.plan(worlds, cfg, solver=engine.SOLVER_COLORED_F32, **kw)
    assert st == 0, msg
    r = {x["name"]: x["workgroups"] for x in rows}
    assert r["k_colour"] == r["k_sweep_colours"]
    return r["k_colour"] - len(worlds)


# the sizes of the one-workgroup colouring: in LDS, its priorities and masks
# in LDS, its priorities alone, none of it (bodies without the floor)
@pytest.mark.parametrize("n,threads", [(MIN_BODIES, 256), (MIN_BODIES, 1024), (24000, 1024),
                                       (30000, 512), (45000, 1024)])
def test_shared_world_equals_its_copies(n, threads):
    w = _world(n)
    cfg = scenes.SceneConfig(iterations=3)
    groups = min(-(-w.n // GROUP_BODIES), MAX_GROUPS)
    copies = MAX_GROUPS * GROUP_MAX // w.n + 1
    assert _shared([w], cfg, solver_threads=threads) == groups - 1
    assert _shared([w] * copies, cfg, solver_threads=threads) == 0
    out = []
    for worlds in ([w], [w] * copies):
        print(f"shared world: {n} bodies, {threads} lanes, {len(worlds)} worlds", flush=True)
        b = engine.make_batch(worlds, cfg, solver=engine.SOLVER_COLORED_F32,
                              solver_threads=threads)
        for graph in (False, True):
            b.step_async(8, use_graph=graph)
            b.sync()
            assert b.stats()["flags"] == 0
        out.append((b.bodies(0), b.contacts(0)["lam"]))
        b.close()
    assert np.array_equal(out[0][0].view(np.uint64), out[1][0].view(np.uint64))
    assert len(out[0][1]) > 0 and np.array_equal(out[0][1].view(np.uint64),
                                                 out[1][1].view(np.uint64))


@pytest.mark.parametrize("iterations", [0, 1, 5])
def test_shared_worlds_of_several_sizes(orc, iterations):
    """Two worlds on several workgroups, the smaller with fewer, and two small
    ones, in an order that is not that of their sizes."""
    worlds = [_world(300, 1, 20), _world(2600, 2, 40), _world(40, 3, 8), _world(7000, 4, 100)]
    cfg = scenes.SceneConfig(iterations=iterations)
    print(f"shared worlds: {iterations} iterations", flush=True)
    assert _shared(worlds, cfg) == 2 * 110 - 2
    _colored_vs_restatement(orc, worlds, cfg, steps=6, every=3)


@pytest.mark.parametrize("boxes", [16, 31, 32, 60])
def test_shared_world_with_a_plank(orc, boxes):
    """A plank lying on a row of boxes: as many manifolds on one body as a
    shared world's lists hold (32), one more, and colours past the 16 that
    are chosen by what is free."""
    b = scenes._Builder()
    b.add(scenes.rectangle_vertices(400.0, 1.0), (0.0, -0.5), mu=0.5)
    for k in range(boxes):
        b.add_dynamic(scenes.rectangle_vertices(1.0, 1.0), (1.5 * k, 0.49), mu=0.5)
    b.add_dynamic(scenes.rectangle_vertices(1.5 * boxes + 1.0, 1.0), (0.75 * (boxes - 1), 1.48), mu=0.5)
    for k in range(MIN_BODIES):
        b.add_dynamic(scenes.rectangle_vertices(0.8, 0.8), (-20.0 - 0.79 * (k % 150), 0.39 + 0.79 * (k // 150)),
                      mu=0.4)
    w, cfg = b.build(), scenes.SceneConfig(iterations=4)
    print(f"plank on {boxes} boxes", flush=True)
    assert _shared([w], cfg) > 0
    _colored_vs_restatement(orc, [w], cfg, steps=12, every=4)


def test_shared_world_without_contacts(orc):
    """Pairs but no manifold (boxes on their corners whose bounds overlap), in
    memory that a world full of contacts has just left."""
    b = engine.make_batch([_world(4000)], scenes.SceneConfig(), solver=engine.SOLVER_COLORED_F32)
    b.step(20)
    b.close()
    b = scenes._Builder()
    b.add(scenes.rectangle_vertices(200.0, 1.0), (0.0, -5.0), mu=0.5)
    for k in range(MIN_BODIES):
        x, y = k % 64, k // 64
        b.add_dynamic(scenes.rectangle_vertices(1.0, 1.0), (0.75 * x, 1.5 * y + 0.75 * (x % 2)),
                      theta=np.pi / 4)
    w, cfg = b.build(), scenes.SceneConfig(iterations=2)
    assert _shared([w], cfg) > 0
    print("pairs without contacts", flush=True)
    gpu = engine.make_batch([w], cfg, solver=engine.SOLVER_COLORED_F32)
    gpu.step(1)
    st = gpu.stats()
    assert st["pairs"] > MIN_BODIES and st["contacts"] == 0 and st["manifolds"] == 0
    gpu.close()
    _colored_vs_restatement(orc, [w], cfg, steps=2, every=1)


def test_shared_world_reports_overflow():
    """Contacts beyond the capacity: the records that touch nothing still take
    their turns, so the step ends and reports the overflow."""
    w, cfg = _world(4000), scenes.SceneConfig(iterations=3)
    b = engine.make_batch([w], cfg, solver=engine.SOLVER_COLORED_F32, max_pairs_per_body=1)
    with pytest.raises(engine.ShapesError):
        b.step(4)
    b.close()
