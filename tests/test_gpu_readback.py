"""Readbacks through the pinned memory: the same rows as array-by-array
copies, for worlds below and above its size, of one world among several."""
import ctypes as C

import numpy as np
import pytest

from shapes_amd import engine, scenes

pytestmark = pytest.mark.gpu


def by_column(b, world):
    """The same state, one column a call."""
    n = b.sizes[world]
    out = np.empty((n, 6))
    for k in range(6):
        col = np.empty(n)
        p = [None] * 6
        p[k] = col.ctypes.data
        engine._check(b._L.shp_batch_read_bodies(b._h, world, *p))
        out[:, k] = col
    return out


@pytest.mark.parametrize("counts", [(1, 7, 300), (21000, 40, 23000)])
def test_readback_columns_agree(counts):
    rng = np.random.Generator(np.random.Philox(5))
    worlds = [scenes.grid_world(rng, n, max(2, int(n ** 0.5)), 1.3, 0.9, 0.0) for n in counts]
    b = engine.make_batch(worlds, scenes.SceneConfig(iterations=2))
    b.step(2)
    for k in range(len(worlds)):
        print(f"readback: world {k} of {b.sizes[k]} bodies", flush=True)
        bodies = b.bodies(k)
        assert np.isfinite(bodies).all() and bodies[1:, 4].any()
        assert np.array_equal(bodies, by_column(b, k))
        c, (slots, boxes) = b.contacts(k), b.aabbs(k)
        n = C.c_int32()
        lam = np.empty((len(c["keys"]), 2))  # the lagrangians alone: another row size
        if len(lam):
            engine._check(b._L.shp_batch_read_contacts(b._h, k, C.byref(n), None, None, None,
                                                       lam.ctypes.data_as(C.POINTER(C.c_double)),
                                                       None))
            assert n.value == len(lam) and np.array_equal(lam, c["lam"])
        assert len(slots) == b.sizes[k] and (boxes[:, 0] <= boxes[:, 1]).all()
    b.close()


def test_non_finite_body_reported_without_a_step():
    w = scenes.random_world(3, count=8)
    w.vx[3] = np.nan
    b = engine.make_batch([w], scenes.SceneConfig())
    with pytest.raises(engine.ShapesError) as e:
        b.sync()
    assert e.value.status == 6
    b.close()
