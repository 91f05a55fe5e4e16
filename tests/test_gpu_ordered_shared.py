"""Worlds that several workgroups solve in the drop-in order, against the
oracle: every bit."""
import numpy as np
import pytest

from shapes_amd import engine, scenes

pytestmark = pytest.mark.gpu

MIN_BODIES = 3072


def _world(n, seed=78, cols=200, y0=1.0):
    rng = np.random.Generator(np.random.Philox(seed))
    return scenes.grid_world(rng, n, cols=cols, spacing=1.05, y0=y0, square_frac=0.5, vel=0.3)


def _check(orc, worlds, cfg, steps, shared=True, **kw):
    st, msg, _, rows = engine.plan(worlds, cfg, **kw)
    assert st == 0 and ("k_solve_flow" in [r["name"] for r in rows]) == shared, msg
    gpu = engine.make_batch(worlds, cfg, **kw)
    refs = [orc.OracleEngine(w, cfg) for w in worlds]
    for s in range(steps):
        print(f"step {s}", flush=True)
        gpu.step_async(2, use_graph=s % 2 == 1)
        gpu.sync()
        assert gpu.stats()["flags"] == 0
        for k, r in enumerate(refs):
            r.step(2)
            assert np.array_equal(gpu.bodies(k).view(np.uint64), r.bodies().view(np.uint64)), (s, k)
            assert np.array_equal(gpu.contacts(k)["lam"].view(np.uint64),
                                  r.contacts()["lam"].view(np.uint64)), (s, k)
    n = gpu.stats()["contacts"]
    gpu.close()
    return n


@pytest.mark.parametrize("iterations", [0, 1, 7])
def test_shared_worlds_of_several_sizes(orc, iterations):
    worlds = [_world(300, 1, 20), _world(3300, 2, 40), _world(40, 3, 8), _world(6000, 4, 80)]
    assert _check(orc, worlds, scenes.SceneConfig(iterations=iterations), 4) > 0


@pytest.mark.parametrize("n,shared", [(MIN_BODIES - 1, False), (MIN_BODIES, True)])
def test_smallest_shared_world(orc, n, shared):  # and the floor
    _check(orc, [_world(n, 5, 30)], scenes.SceneConfig(iterations=4), 4, shared)


@pytest.mark.parametrize("boxes", [31, 32, 33])
def test_plank_of_as_many_manifolds_as_lists_hold(orc, boxes):
    """With bounce on some boxes, so both forms of the items."""
    b = scenes._Builder()
    b.add(scenes.rectangle_vertices(400.0, 1.0), (0.0, -0.5), mu=0.5, bounce=0.3)
    for k in range(boxes):
        b.add_dynamic(scenes.rectangle_vertices(1.0, 1.0), (1.5 * k, 0.49), mu=0.5, bounce=0.4 * (k % 2))
    b.add_dynamic(scenes.rectangle_vertices(1.5 * boxes + 1.0, 1.0), (0.75 * (boxes - 1), 1.48), mu=0.5,
                  bounce=0.2)
    for k in range(MIN_BODIES):
        b.add_dynamic(scenes.rectangle_vertices(0.8, 0.8),
                      (-20.0 - 0.79 * (k % 150), 0.39 + 0.79 * (k // 150)), mu=0.4)
    assert _check(orc, [b.build()], scenes.SceneConfig(iterations=4), 3) > 2 * boxes


def test_contacts_beyond_the_capacity_are_reported():
    w, cfg = _world(4000), scenes.SceneConfig(iterations=3)
    b = engine.make_batch([w], cfg, max_pairs_per_body=1)
    with pytest.raises(engine.ShapesError):
        b.step(4)
    b.close()
