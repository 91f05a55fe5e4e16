"""The coloured sweeps' workgroups as the plan has them (no GPU): the small
worlds' launch holds wavefronts for larger ones only when there are any."""
import pytest

from shapes_amd import engine, scenes


@pytest.mark.parametrize("sizes,lanes", [((8, 64, 256), 256), ((256,) * 9, 256), ((257,), 1024),
                                         ((8, 257, 40), 1024), ((1088, 3), 1024), ((1089, 200), 256)])
def test_lanes_of_the_small_worlds(sizes, lanes):
    worlds = [scenes.random_world(k, count=n - 1, cols=max(4, int(n ** 0.5)))
              for k, n in enumerate(sizes)]
    st, msg, _, rows = engine.plan(worlds, scenes.SceneConfig(), solver=engine.SOLVER_COLORED_F32,
                                   solver_threads=64)
    assert st == 0, msg
    r = {x["name"]: x for x in rows}["k_sweep_waves"]
    assert r["workgroup_size"] == lanes
    assert r["workgroups"] == -(-sum(n <= 1088 for n in sizes) // 4)
