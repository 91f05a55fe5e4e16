"""Which broadphase a batch gets by default (host only): the grid for large
worlds or for many pairs of bodies in all."""
import numpy as np
import pytest

from shapes_amd import engine, scenes


def _world(bodies):  # the floor among them
    rng = np.random.Generator(np.random.Philox(4))
    return scenes.grid_world(rng, bodies - 1, cols=40, spacing=1.05, y0=1.0, square_frac=0.5)


@pytest.mark.parametrize("bodies,worlds,grid", [(1536, 1, False), (1537, 1, True),
                                                (1000, 6, False), (1000, 7, True),
                                                (100, 600, False), (100, 601, True), (8, 64, False)])
def test_default_broadphase(bodies, worlds, grid):
    st, msg, p, _ = engine.plan([_world(bodies)] * worlds, scenes.SceneConfig())
    assert st == 0, msg
    assert (p["broadphase"] == engine.BROADPHASE_GRID) == grid
