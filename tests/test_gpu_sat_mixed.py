"""SAT of hulls of 3 to 8 vertices and circles side by side in a wavefront, at
the edges of its 64 pairs, against the oracle, bit for bit."""
import numpy as np
import pytest

from shapes_amd import engine, scenes

pytestmark = pytest.mark.gpu


def _ngon(n, r):
    t = 2 * np.pi * (np.arange(n) + 0.25) / n
    return list(zip(r * np.cos(t), r * np.sin(t)))


def _row(pairs, circles, fill=140):
    """`pairs` bodies in a row, each overlapping the next, hulls of 3..8
    vertices (every seventh a circle), and bodies apart from all, so that the
    world is too large for the small worlds' path."""
    b = scenes._Builder()
    for k in range(pairs + 1):
        at = (0.9 * k, 0.05 * (k % 3))
        if circles and k % 7 == 3:
            b.add_circle(0.5, at, mass=1.0, inertia=0.125, mu=0.3)
        else:
            b.add_dynamic(_ngon(3 + (5 * k) % 6, 0.6), at, theta=0.1 * k, mu=0.3)
    for k in range(fill):
        b.add_dynamic(_ngon(3 + k % 6, 0.4), (3.0 * k, 50.0), mu=0.3)
    return b.build()


def _same(a, b):
    a, b = np.ascontiguousarray(a), np.ascontiguousarray(b)
    return a.dtype == b.dtype and a.shape == b.shape and a.tobytes() == b.tobytes()


def _compare(orc, w, cfg, steps, **kw):
    gpu, ref = engine.make_batch([w], cfg, **kw), orc.OracleEngine(w, cfg)
    seen = 0
    for s in range(steps):
        gpu.step(1)
        ref.step(1)
        a, b = gpu.contacts(0), ref.contacts()
        for k in ("keys", "flip", "geom", "lam"):
            assert _same(a[k], b[k]), (s, k)
        assert _same(gpu.bodies(0), ref.bodies()), s
        seen = max(seen, len(b["keys"]))
    gpu.close()
    return seen


@pytest.mark.parametrize("circles", [False, True])
@pytest.mark.parametrize("pairs", [1, 2, 63, 64, 65, 127, 129, 257])
def test_wavefronts_match_the_oracle(orc, pairs, circles):
    print(f"{pairs} pairs, circles {circles}", flush=True)
    cfg = scenes.SceneConfig(iterations=2, gy=0.0)
    w = _row(pairs, circles)
    st, msg, _, rows = engine.plan([w], cfg)
    assert st == 0 and "k_sat" in [r["name"] for r in rows], msg
    assert _compare(orc, w, cfg, steps=3) >= pairs
