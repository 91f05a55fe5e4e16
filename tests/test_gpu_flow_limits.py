"""Worlds solved by several workgroups where that path ends: colours past its
limit, told by one workgroup while others of the world still start."""
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
