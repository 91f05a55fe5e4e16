"""What the flags report, and when: an overflow in a step that is not the last
of its call, over every broadphase, and the one of the front in one launch."""
import numpy as np
import pytest

from shapes_amd import engine, scenes

pytestmark = pytest.mark.gpu

PAIR_OVERFLOW = 1
LIMIT = 128  # bodies of the front in one launch, floors among them


def _burst(n, seed, speed):
    """n boxes on one spot (all pairs of them), each with a direction of its
    own: two steps on they are apart."""
    rng = np.random.default_rng(seed)
    b = scenes._Builder()
    b.add(scenes.rectangle_vertices(40.0, 1.0), (0.0, -500.0), mu=0.5)
    for k in range(n):
        a = 2 * np.pi * k / n
        b.add_dynamic(scenes.rectangle_vertices(1.0, 0.9),
                      (0.3 * np.cos(a) + rng.uniform(-0.05, 0.05), 0.3 * np.sin(a)), theta=a,
                      vel=(speed * np.cos(a), speed * np.sin(a)))
    return b.build()


CASES = [(LIMIT - 1, engine.BROADPHASE_AUTO, engine.SOLVER_ORDERED_F64),
         (200, engine.BROADPHASE_SCAN, engine.SOLVER_ORDERED_F64),
         (200, engine.BROADPHASE_SCAN, engine.SOLVER_COLORED_F32),
         (200, engine.BROADPHASE_GRID_16, engine.SOLVER_ORDERED_F64),
         (200, engine.BROADPHASE_GRID_1, engine.SOLVER_COLORED_F32)]


@pytest.mark.parametrize("n,broadphase,solver", CASES)
def test_an_early_overflow_is_reported(n, broadphase, solver):
    kw = dict(max_pairs_per_body=1, broadphase=broadphase, solver=solver)
    w, cfg = _burst(n, 3, 4e4), scenes.SceneConfig(iterations=1)
    cap = w.n + 1024
    _, _, _, rows = engine.plan([w], cfg, **kw)
    assert ("k_front_small" in [r["name"] for r in rows]) == (w.n <= LIMIT)
    print(f"{n} boxes, broadphase {broadphase}, solver {solver}", flush=True)
    b = engine.make_batch([w], cfg, **kw)
    with pytest.raises(engine.ShapesError, match="capacity exceeded"):
        b.step(1)
    st = b.stats()
    assert st["flags"] & PAIR_OVERFLOW and st["pairs"] == cap
    b.close()
    b = engine.make_batch([w], cfg, **kw)
    b.step_async(2)
    b.step_async(2, use_graph=True)
    with pytest.raises(engine.ShapesError, match="capacity exceeded"):
        b.sync()
    st = b.stats()
    assert st["pairs"] < cap and st["flags"] & PAIR_OVERFLOW
    b.close()


def test_the_overflow_of_the_front_keeps_the_first_pairs():
    """The pairs below the capacity are those of the separate launches."""
    cfg, out = scenes.SceneConfig(iterations=1), []
    w = _burst(LIMIT - 1, 5, 0.0)
    for broadphase in (engine.BROADPHASE_SCAN, engine.BROADPHASE_GRID):
        b = engine.make_batch([w], cfg, max_pairs_per_body=1, broadphase=broadphase)
        print(f"broadphase {broadphase}", flush=True)
        with pytest.raises(engine.ShapesError, match="capacity exceeded"):
            b.step(1)
        out.append((b.pairs(), b.contacts()["keys"]))
        b.close()
    pairs = out[0][0]
    assert len(pairs) == w.n + 1024 and len(out[0][1]) > 0
    # a body's pairs that straddle the capacity: the grid keeps as many of them
    first = pairs[:, 0] > pairs[-1, 0]
    assert np.array_equal(pairs[first], out[1][0][:first.sum()])
    keys = out[0][1][out[0][1][:, 0] > pairs[-1, 0]]
    assert np.array_equal(keys, out[1][1][:len(keys)])


def test_flags_outlive_a_new_layout():
    """An unread overflow is still reported after an append that lays the
    batch out again."""
    w = _burst(60, 3, 4e4)
    w.capacity = w.n + 1
    b = engine.make_batch([w], scenes.SceneConfig(iterations=1), max_pairs_per_body=1)
    print("append after an overflow", flush=True)
    b.step_async(3)
    b.append(0, 100.0, 100.0, hull=scenes.rectangle_vertices(1.0, 1.0))
    b.step_async(1)
    with pytest.raises(engine.ShapesError, match="capacity exceeded"):
        b.sync()
    b.close()
