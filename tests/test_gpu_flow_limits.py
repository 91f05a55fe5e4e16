"""Worlds solved by several workgroups where that path ends: colours past its
limit, fewer workgroups than wanted, records that fill a workgroup's LDS, waits
that give up; and batches that they share the GPU or the launch with."""
import ctypes as C

import numpy as np
import pytest

from shapes_amd import engine, scenes
from test_gpu_colored import _colored_vs_restatement

pytestmark = pytest.mark.gpu

MIN_BODIES = 2048


def _planks(n, boxes, seed):
    """Planks, each on `boxes` boxes (as many manifolds on one body), in a
    field of single boxes that makes the world one of `n` bodies or more."""
    rng = np.random.default_rng(seed)
    b = scenes._Builder()
    b.add(scenes.rectangle_vertices(4000.0, 1.0), (0.0, -0.5), mu=0.5)
    x = 0.0
    for k in boxes:
        for q in range(k):
            b.add_dynamic(scenes.rectangle_vertices(1.0, 1.0), (x + 1.5 * q, 0.49), mu=0.5)
        b.add_dynamic(scenes.rectangle_vertices(1.5 * k + 1.0, 1.0), (x + 0.75 * (k - 1), 1.48), mu=0.5)
        x += 1.5 * k + 4.0
    for k in range(n):
        b.add_dynamic(scenes.rectangle_vertices(0.8, 0.8),
                      (-20.0 - 0.79 * (k % 150), 0.39 + 0.79 * (k // 150)), mu=0.4,
                      vel=(0.1 * rng.uniform(-1, 1), 0.0))
    return b.build()


def test_colours_past_the_limit(orc):
    """17 to 31 manifolds on one body take colours past 32: the workgroup that
    finds one says so, and one workgroup colours the world instead, whatever
    the others have seen of it."""
    worlds = [_planks(MIN_BODIES + 500 * k, [17 + k, 24, 31 - k, 20], k) for k in range(3)]
    cfg = scenes.SceneConfig(iterations=2)
    st, msg, _, rows = engine.plan(worlds, cfg, solver=engine.SOLVER_COLORED_F32)
    assert st == 0 and {r["name"]: r["workgroups"] for r in rows}["k_colour"] > 3, msg
    print("colours past the limit", flush=True)
    _colored_vs_restatement(orc, worlds, cfg, steps=16, every=4)
    b = engine.make_batch(worlds, cfg, solver=engine.SOLVER_COLORED_F32)
    b.step(4)
    assert b.stats()["flags"] == 0 and b.stats()["max_levels"] > 32
    b.close()


@pytest.mark.parametrize("sizes", [(256, 2, 255, 90, 17), (3,), (1200, 250, 40)])
def test_small_worlds_without_larger_ones(orc, sizes):
    """The small worlds' sweeps when none of them takes more than a wavefront,
    alone and beside a world with a workgroup of its own."""
    worlds = [scenes.random_world(50 + k, count=n - 1, cols=max(4, int(n ** 0.5)))
              for k, n in enumerate(sizes)]
    print(f"worlds of {sizes} bodies", flush=True)
    _colored_vs_restatement(orc, worlds, scenes.SceneConfig(iterations=5), steps=40, every=20, threads=64)


def _pile(n, seed=78, cols=60):
    rng = np.random.Generator(np.random.Philox(seed))
    return scenes.grid_world(rng, n, cols=cols, spacing=1.05, y0=1.0, square_frac=0.5, vel=0.3)


def _limit(batch, seats=1 << 29, polls=1 << 20):
    f = batch._L.shp_batch_flow_limits  # for tests: not in the header
    f.argtypes = [C.c_void_p, C.c_int32, C.c_int32]
    assert f(batch._h, seats, polls) == 0


def _bits(worlds, cfg, steps, limit=None, **kw):
    b = engine.make_batch(worlds, cfg, **kw)
    if limit is not None:
        _limit(b, seats=limit)
    for k in range(2):
        b.step_async(steps, use_graph=k == 1)
        b.sync()
        assert b.stats()["flags"] == 0
    out = [(b.bodies(k).view(np.uint64), b.contacts(k)["lam"].view(np.uint64)) for k in range(len(worlds))]
    b.close()
    return out


@pytest.mark.parametrize("solver", [engine.SOLVER_ORDERED_F64, engine.SOLVER_COLORED_F32])
@pytest.mark.parametrize("n,n2", [(4096, 3300), (20000, 3300)])
def test_fewer_workgroups_than_wanted(solver, n, n2):
    """As many workgroups join as a busy GPU has room for: the ordered solver
    leaves the world to one, the coloured colours and sweeps it with those,
    or with one when their records do not fit in LDS."""
    worlds, cfg = [_pile(n), _pile(30, 5, 8), _pile(n2, 4)], scenes.SceneConfig(iterations=3)
    st, msg, _, rows = engine.plan(worlds, cfg, solver=solver)
    r = {x["name"]: x["workgroups"] for x in rows}
    assert st == 0 and (r.get("k_solve_flow", 0) > 40 or r["k_colour"] > 40), msg
    want = _bits(worlds, cfg, 6, solver=solver)
    for seats in (1, 2, 7, 33):
        print(f"{n} bodies, solver {solver}, {seats} seats", flush=True)
        got = _bits(worlds, cfg, 6, limit=seats, solver=solver)
        for (a, b), (x, y) in zip(want, got):
            assert len(b) and np.array_equal(a, x) and np.array_equal(b, y), seats


@pytest.mark.parametrize("solver", [engine.SOLVER_ORDERED_F64, engine.SOLVER_COLORED_F32])
def test_a_wait_that_gives_up_is_reported(solver):
    """A workgroup that leaves its world after it was counted in (the waits end
    at once here): the others' waits end too, and the step says so."""
    b = engine.make_batch([_pile(4096)], scenes.SceneConfig(iterations=2), solver=solver)
    _limit(b, polls=0)
    print(f"waits that give up, solver {solver}", flush=True)
    with pytest.raises(engine.ShapesError, match="wait between workgroups"):
        b.step(1)
    assert b.stats()["flags"] & 16
    b.close()


def test_batches_on_the_gpu_at_once():
    """Batches whose shared worlds want every CU, stepped on their streams at
    the same time."""
    cfg = scenes.SceneConfig(iterations=3)
    kinds = [(engine.SOLVER_COLORED_F32, 24000), (engine.SOLVER_ORDERED_F64, 12000),
             (engine.SOLVER_COLORED_F32, 16000)]
    want = [_bits([_pile(n)], cfg, 6, solver=s) for s, n in kinds]
    print("three batches at once", flush=True)
    bs = [engine.make_batch([_pile(n)], cfg, solver=s) for s, n in kinds]
    for k in range(12):
        for b in bs:
            b.step_async(1, use_graph=k >= 6)
    for b, ((x, lam),) in zip(bs, want):
        b.sync()
        assert b.stats()["flags"] == 0
        assert np.array_equal(b.bodies(0).view(np.uint64), x)
        assert np.array_equal(b.contacts(0)["lam"].view(np.uint64), lam)
        b.close()


def test_shared_world_beside_small_worlds_sweeps(orc):
    """solver_threads 64 with a world for several workgroups, one for one, and
    small ones of both forms."""
    worlds = [scenes.random_world(60, count=300, cols=18), _pile(2600, 2, 40),
              scenes.random_world(61, count=40), _pile(1500, 3, 30)]
    print("shared, single and small worlds", flush=True)
    _colored_vs_restatement(orc, worlds, scenes.SceneConfig(iterations=4), steps=8, every=4, threads=64)


@pytest.mark.parametrize("solver", [engine.SOLVER_ORDERED_F64, engine.SOLVER_COLORED_F32])
@pytest.mark.parametrize("seats", [1 << 29, 3])
def test_solve_profile_of_a_shared_world(solver, seats):
    """The solve's sub-phases are timed whoever solves the largest world, which
    is the second here."""
    b = engine.make_batch([_pile(40, 3, 8), _pile(5000)], scenes.SceneConfig(iterations=6), solver=solver)
    _limit(b, seats=seats)
    b.step(10)
    b.set_timing(True)
    print(f"solve profile, solver {solver}, {seats} seats", flush=True)
    b.step(20)
    us, ms = b.solve_profile(), b.timing()
    b.close()
    assert us[3] > 5 and us[0] > 0
    coloured = solver == engine.SOLVER_COLORED_F32
    assert us[3] + us[4] <= 1e3 * ms["sweeps"] + 1
    if coloured:
        assert us[0] <= 1e3 * ms["colouring"] + 1
