"""The step's front in one launch, at the edges of its range (128 bodies in
all; 512 pairs to a round) and with several worlds, circles, empty slots and
the learned start, against the oracle and against the separate launches."""
import numpy as np
import pytest

from shapes_amd import engine, scenes

pytestmark = pytest.mark.gpu

LIMIT = 128  # bodies, floors among them


def _names(worlds, cfg):
    st, msg, _, rows = engine.plan(worlds, cfg)
    assert st == 0, msg
    return [r["name"] for r in rows]


def _clump(n, seed):
    """n boxes in a heap: more pairs than bodies."""
    rng = np.random.default_rng(seed)
    b = scenes._Builder()
    b.add(scenes.rectangle_vertices(40.0, 1.0), (0.0, -0.5), mu=0.5)
    side = max(2.0, 0.55 * n ** 0.5)
    for k in range(n):
        b.add_dynamic(scenes.rectangle_vertices(1.0, 0.8), (rng.uniform(-side, side), rng.uniform(0.4, side)),
                      theta=rng.uniform(0, 3), mu=0.4)
    return b.build()


@pytest.mark.parametrize("sizes,small", [((1,), True), ((2, 3), True), ((31, 32, 33), True),
                                         ((LIMIT - 1,), True), ((LIMIT - 3, 1), True), ((LIMIT,), False)])
def test_front_matches_the_oracle(orc, sizes, small):
    worlds = [_clump(n, 7 + n) for n in sizes]  # and a floor each
    cfg = scenes.SceneConfig(iterations=3)
    print(f"front of {sizes} boxes", flush=True)
    assert ("k_front_small" in _names(worlds, cfg)) == small
    gpu = engine.make_batch(worlds, cfg, max_pairs_per_body=32)
    refs = [orc.OracleEngine(w, cfg) for w in worlds]
    for s in range(6):
        gpu.step_async(1, use_graph=s > 2)
        gpu.sync()
        assert gpu.stats()["flags"] == 0
        for k, r in enumerate(refs):
            r.step(1)
            assert np.array_equal(gpu.bodies(k).view(np.uint64), r.bodies().view(np.uint64)), (s, k)
            a, b = gpu.contacts(k), r.contacts()
            assert np.array_equal(a["lam"].view(np.uint64), b["lam"].view(np.uint64)), (s, k)
    gpu.close()


@pytest.mark.parametrize("warm", [engine.WARM_ZERO, engine.WARM_LEARNED])
def test_front_equals_the_separate_launches(warm):
    """The same scene beside a batch too large for the one launch (whose first
    world it is), with circles, the overlays' probe and both warm starts."""
    from shapes_amd import warmstart
    scene = scenes.balls(dims=(8, 8)).worlds[0]
    cfg = scenes.SceneConfig(iterations=3)
    assert "k_front_small" in _names([scene], cfg) and "k_front_small" not in _names([scene] * 5, cfg)
    out = []
    for n in (1, 5):
        print(f"{n} worlds, warm start {warm}", flush=True)
        b = engine.make_batch([scene] * n, cfg, warm_start=warm)
        if warm == engine.WARM_LEARNED:
            b.set_mlp(np.load(warmstart.DEFAULT_MODEL))
        for _ in range(30):
            b.step(1)
        b.probe_contacts()
        out.append((b.bodies(0), b.contacts(0)))
        st = b.stats()
        assert st["flags"] == 0
        out[-1] += ((st["pairs"] / n, st["contacts"] / n),)
        b.close()
    assert np.array_equal(out[0][0].view(np.uint64), out[1][0].view(np.uint64))
    for key in out[0][1]:
        assert np.array_equal(out[0][1][key], out[1][1][key]), key
    assert out[0][2] == out[1][2]


def test_pair_overflow_is_reported():
    b = engine.make_batch([_clump(200, 3)], scenes.SceneConfig(), max_pairs_per_body=1)
    n = b.stats()
    try:
        b.step(1)
        assert b.stats()["pairs"] <= 201 + 1024
    except engine.ShapesError:
        pass
    b.close()
