"""The grid broadphase's rows of cells against the scan of every pair: the same
pairs, so the same contacts and bodies, bit for bit."""
import numpy as np
import pytest

from shapes_amd import engine, scenes

pytestmark = pytest.mark.gpu


def _boxes(xy, half=0.5, floor=True):
    b = scenes._Builder()
    if floor:
        b.add(scenes.rectangle_vertices(50.0, 1.0), (float(np.mean([p[0] for p in xy])),
                                                     min(p[1] for p in xy) - 1.01), mu=0.5)
    for k, (x, y) in enumerate(xy):
        b.add_dynamic(scenes.rectangle_vertices(2 * half, 2 * half * (0.5 + 0.5 * ((k * 7) % 5) / 4)),
                      (float(x), float(y)), theta=0.1 * (k % 9), mu=0.4)
    return b.build()


def _worlds():
    rng = np.random.default_rng(3)
    grid = [(1.02 * (k % 12), 1.02 * (k // 12)) for k in range(120)]
    return {
        "clump of more partners than are kept": _boxes(rng.uniform(0, 3.0, (40, 2))),
        "column longer than its table": _boxes([(0.0, 1.01 * k) for k in range(70)]),
        "row across the table's end": _boxes([(1.01 * k - 40.0, 0.0) for k in range(80)]),
        "negative cells": _boxes([(x - 500.0, y - 700.0) for x, y in grid]),
        "far out": _boxes([(x + 3.0e8, y + 2.0e8) for x, y in grid]),
        "where a box's bounds round to more than a cell": _boxes(
            [(x * 4 + 4.0e15, y * 4 + 4.0e15) for x, y in grid], floor=False),
        "three bodies": _boxes([(0.0, 0.0), (0.9, 0.2), (0.4, 1.0)]),
    }


@pytest.mark.parametrize("name", list(_worlds()))
def test_rows_find_the_scanned_pairs(name):
    w, cfg = _worlds()[name], scenes.SceneConfig(iterations=2)
    out = []
    for bp in (engine.BROADPHASE_SCAN, engine.BROADPHASE_GRID_1, engine.BROADPHASE_GRID_16):
        print(f"{name}: broadphase {bp}", flush=True)
        b = engine.make_batch([w, w], cfg, broadphase=bp, max_pairs_per_body=64)
        b.step(3)
        out.append((b.stats()["pairs"], b.bodies(1), b.contacts(1)["lam"]))
        b.close()
    for pairs, bodies, lam in out[1:]:
        assert pairs == out[0][0]
        assert np.array_equal(bodies.view(np.uint64), out[0][1].view(np.uint64))
        assert np.array_equal(lam.view(np.uint64), out[0][2].view(np.uint64))
