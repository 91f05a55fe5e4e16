"""Small worlds' coloured sweeps at the edges of their forms: one wavefront up
to 256 bodies, four above, a workgroup of its own above 1088; workgroups that
hold both forms, and the last one partly empty.  Every bit of the oracle's."""
import numpy as np
import pytest

from shapes_amd import engine, scenes
from test_gpu_colored import _colored_vs_restatement

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,own", [((256, 257), 0), ((257, 258, 20, 5, 255), 0),
                                       ((1088, 1089, 1087), 1), ((600, 12, 300, 11, 900, 10, 9), 0)])
def test_sweep_forms(orc, sizes, own):
    worlds = [scenes.random_world(40 + k, count=n - 1, cols=max(4, int(n ** 0.5)))
              for k, n in enumerate(sizes)]
    assert [w.n for w in worlds] == list(sizes)
    cfg = scenes.SceneConfig(iterations=5)
    st, msg, _, rows = engine.plan(worlds, cfg, solver=engine.SOLVER_COLORED_F32, solver_threads=64)
    names = {r["name"]: r["workgroups"] for r in rows}
    assert st == 0 and names.get("k_sweep_colours", 0) == own, msg
    assert names["k_sweep_waves"] == (len(sizes) - own + 3) // 4
    print(f"worlds of {sizes} bodies", flush=True)
    _colored_vs_restatement(orc, worlds, cfg, steps=60, every=20, threads=64)
