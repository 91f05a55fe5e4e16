"""Contact generation's tiles of 256 pairs, a lane to a contact: boxes standing
on a floor, two contacts each, beside the oracle, bit for bit."""
import numpy as np
import pytest

from shapes_amd import engine, scenes
from test_gpu_colored import _colored_vs_restatement

pytestmark = pytest.mark.gpu


def _row(n, corner=0):
    """n boxes flat on a floor, the first `corner` of them on a corner (one
    contact)."""
    b = scenes._Builder()
    b.add(scenes.rectangle_vertices(4.0 * n + 10.0, 1.0), (0.0, -0.5), mu=0.5)
    for k in range(n):
        x = 2.0 * (k - n / 2)
        if k < corner:
            b.add_dynamic(scenes.rectangle_vertices(1.0, 1.0), (x, 0.7), theta=np.pi / 4, mu=0.5)
        else:
            b.add_dynamic(scenes.rectangle_vertices(1.0, 1.0), (x, 0.49), mu=0.5)
    return b.build()


@pytest.mark.parametrize("n,corner", [(1, 0), (128, 0), (129, 0), (255, 3), (256, 0), (257, 1),
                                      (512, 512), (513, 0)])
def test_rows_of_boxes_match(orc, n, corner):
    w, cfg = _row(n, corner), scenes.SceneConfig(iterations=3)
    print(f"row of {n} boxes, {corner} on a corner", flush=True)
    _colored_vs_restatement(orc, [w], cfg, steps=4, every=2)
    gpu, ref = engine.make_batch([w], cfg), orc.OracleEngine(w, cfg)
    for _ in range(3):
        gpu.step(1)
        ref.step(1)
        assert np.array_equal(gpu.bodies(0).view(np.uint64), ref.bodies().view(np.uint64))
        a, b = gpu.contacts(0), ref.contacts()
        assert np.array_equal(a["lam"].view(np.uint64), b["lam"].view(np.uint64))
    st = gpu.stats()
    # boxes apart from each other: a manifold each, flat ones with two contacts
    assert st["manifolds"] == n and st["contacts"] == 2 * n - corner
    assert st["warm_hits"] == st["contacts"]
    gpu.close()


def test_records_of_many_rows(orc):
    """The records that contact generation writes itself (256 worlds, 1024
    lanes): every world as alone."""
    worlds = [_row(1 + k % 5) for k in range(256)]
    cfg = scenes.SceneConfig(iterations=3)
    print("256 rows of boxes", flush=True)
    st, msg, _, rows = engine.plan(worlds, cfg, solver=engine.SOLVER_COLORED_F32, solver_threads=1024)
    assert st == 0 and "k_pack_manifolds" not in [r["name"] for r in rows], msg
    _colored_vs_restatement(orc, worlds, cfg, steps=4, every=4, threads=1024)
