"""The drop-in solver's schedule at the sizes where its storage changes, bit
for bit against the oracle: levels wider than their LDS slots, lagrangians
beyond the LDS pool, links in global memory, chains of one item, no sweeps
and many."""
import numpy as np
import pytest

from shapes_amd import engine, scenes
from test_gpu_parity import compare_state

pytestmark = pytest.mark.gpu

BOX = scenes.rectangle_vertices(1.0, 1.0)


def row(n):
    """n boxes side by side on one floor, not touching: one level of n items."""
    b = scenes._Builder()
    b.add(scenes.rectangle_vertices(3.0 * n, 1.0), (0.0, -0.5), mu=0.5)
    for k in range(n):
        b.add_dynamic(BOX, ((k - n / 2) * 1.5, 0.495), vel=(0.1 * (k % 7), 0.0))
    return b.build()


def wall(cols, rows):
    """A wall of bricks, six neighbours each: about six contacts a body."""
    b = scenes._Builder()
    b.add(scenes.rectangle_vertices(4.0 * cols, 1.0), (0.0, -0.5), mu=0.5)
    for r in range(rows):
        for k in range(cols):
            b.add_dynamic(scenes.rectangle_vertices(2.0, 1.0),
                          ((k - cols / 2) * 1.999 + (r % 2), 0.499 + 0.999 * r),
                          vel=(0.01 * (k % 3), 0.0))
    return b.build()


def column(n):
    b = scenes._Builder()
    b.add(scenes.rectangle_vertices(9.0, 1.0), (0.0, -0.5), mu=0.5)
    for k in range(n):
        b.add_dynamic(BOX, (0.001 * (k % 5), 0.499 + 0.999 * k), bounce=0.3 if k % 4 == 1 else 0.0)
    return b.build()


CASES = [("row", 1020, 256, 3), ("row", 2050, 512, 2), ("row", 192, 0, 0), ("row", 193, 512, 1),
         ("wall", 12, 0, 4), ("wall", 24, 0, 2), ("wall", 24, 256, 2), ("column", 40, 0, 5),
         ("column", 3, 0, 32760), ("column", 2, 512, 40)]


@pytest.mark.parametrize("shape,size,threads,iterations", CASES)
def test_schedule_bitwise(orc, shape, size, threads, iterations):
    print(f"schedule: {shape} {size}, {threads} lanes, {iterations} sweeps", flush=True)
    w = {"row": row, "wall": lambda n: wall(n, n), "column": column}[shape](size)
    cfg = scenes.SceneConfig(iterations=iterations)
    gpu = engine.make_batch([w], cfg, solver_threads=threads)
    ref = orc.OracleEngine(w, cfg)
    for step in range(1, 4 if iterations > 1000 else 9):
        gpu.step(1)
        ref.step(1)
        compare_state(gpu, ref, step)
    assert len(ref.contacts()["keys"]) >= min(size, 2)
    gpu.close()


def test_schedule_of_uneven_worlds_bitwise(orc):
    """One batch of worlds of every kind: narrow, wide, without contacts."""
    worlds = [column(6), row(300), wall(8, 8), column(1), row(1), wall(20, 20)]
    far = column(2)
    far.py[1:] += 50.0
    worlds.append(far)
    cfg = scenes.SceneConfig(iterations=4)
    gpu = engine.make_batch(worlds, cfg)
    refs = [orc.OracleEngine(w, cfg) for w in worlds]
    for step in range(1, 7):
        gpu.step(1)
        for k, r in enumerate(refs):
            r.step(1)
            compare_state(gpu, r, step, world=k)
    gpu.close()
