"""The network's forward pass on device buffers that share memory: the outputs
over the features' own rows, at their start, further in and across their end."""
import ctypes as C

import numpy as np
import pytest

from shapes_amd import engine, warmstart
from test_zz_no_alloc import _check, _hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 17, 5000, 65536])
def test_outputs_over_the_features(n):
    hip = _hip()
    m = engine.Mlp(np.load(warmstart.DEFAULT_MODEL))
    feats = np.random.default_rng(n).normal(size=(n, 14)).astype(np.float32)
    want = m.forward(feats)
    buf = C.c_void_p()
    _check(hip.hipMalloc(C.byref(buf), feats.nbytes + 8 * n))
    # floats from the features' start: over them, and right behind them
    for at in (0, 1, 7 * n, 14 * n - 1, 14 * n):
        print(f"{n} rows, outputs at {at}", flush=True)
        _check(hip.hipMemcpy(buf, feats.ctypes.data, feats.nbytes, 1))
        _check(hip.hipDeviceSynchronize())
        m.forward_noalloc(buf.value, n, buf.value + 4 * at)
        _check(hip.hipDeviceSynchronize())
        got = np.empty((n, 2), dtype=np.float32)
        _check(hip.hipMemcpy(got.ctypes.data, C.c_void_p(buf.value + 4 * at), got.nbytes, 2))
        assert np.array_equal(got.view(np.uint32), want.view(np.uint32)), at
    _check(hip.hipFree(buf))
    m.close()
