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


@pytest.mark.parametrize("solver,threads", [(engine.SOLVER_ORDERED_F64, 0), (engine.SOLVER_COLORED_F32, 64)])
def test_small_worlds_pay_nothing_for_a_large_one(solver, threads):
    """The lines by which several workgroups share a world belong to its own
    bodies: small worlds beside it take the memory that they take alone."""
    large = scenes.random_world(1, count=4095, cols=64)
    small = [scenes.random_world(2, count=63, cols=8)] * 500

    def plan(worlds):
        st, msg, p, rows = engine.plan(worlds, scenes.SceneConfig(), solver=solver, solver_threads=threads,
                                       broadphase=engine.BROADPHASE_GRID)
        assert st == 0, msg
        return p["device_bytes"], {r["name"]: r["workgroups"] for r in rows}

    both, rows = plan([large] + small)
    assert rows.get("k_solve_flow", rows.get("k_colour", 0) - 500) > 20
    alone, of_large = plan(small)[0], plan([large])[0]
    bodies = 500 * 64
    assert both - alone - of_large < 8 * bodies
