"""The network's kernels at the edges of their tiles (16 rows forward, 64 rows
in training, 64 workgroups) against the FP64 reference."""
import numpy as np
import pytest

import mlp_ref as M
from shapes_amd import engine

pytestmark = pytest.mark.gpu


def _data(n, seed):
    rng = np.random.default_rng(seed)
    X = rng.normal(size=(n, 14)).astype(np.float32)
    T = (np.sin(X[:, :2]) + 0.3 * X[:, 2:4]).astype(np.float32)
    return X, T


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 65, 1000, 16384, 16401])
def test_forward_rows(n):
    print(f"forward: {n} rows", flush=True)
    p = M.init_params(5)
    X, _ = _data(n, n)
    net = engine.Mlp(p)
    y = net.forward(X)
    ref, _, _ = M.forward(p, X)
    # BF16 inputs, weights and activations (2^-9 each) through four layers
    assert np.abs(y - ref).max() <= 2e-2 * max(np.abs(ref).max(), 1.0)
    net.close()


@pytest.mark.parametrize("n,huber", [(1, 0.0), (63, 0.0), (64, 0.5), (65, 0.0), (4096, 0.0),
                                     (4097, 0.0), (9000, 0.0)])
def test_gradient_rows(n, huber):
    print(f"gradient: {n} rows", flush=True)
    p = M.init_params(6)
    X, T = _data(n, 40 + n)
    net = engine.Mlp(p)
    net.set_loss(huber)
    g, loss = net.gradient(X, T)
    if huber:  # the Huber gradient: that of targets within huber of the outputs
        y = M.forward(p, X)[0]
        T = (y - np.clip(y - T, -huber, huber)).astype(np.float32)
        gr = M.gradient(p, X, T)[0]
    else:
        gr, lr = M.gradient(p, X, T)
        assert abs(loss - lr) <= 2e-2 * lr
    k = 0
    for name, shape in M.SHAPES:
        m = int(np.prod(shape))
        a, b = g[k:k + m].astype(np.float64), gr[k:k + m]
        assert np.linalg.norm(a - b) <= 5e-2 * np.linalg.norm(b) + 1e-6, name
        k += m
    net.close()


@pytest.mark.parametrize("batch,steps", [(64, 3), (4096, 2), (4160, 2)])
def test_training_steps_follow_the_gradient(batch, steps):
    """Adam on the library's own gradients of the gathered rows, in FP64."""
    print(f"train: {steps} steps of {batch} rows", flush=True)
    X, T = _data(5000, 9)
    idx = np.random.default_rng(1).integers(0, len(X), batch * steps).astype(np.int32)
    net = engine.Mlp(M.init_params(8))
    net.set_data(X, T)
    p = net.params().astype(np.float64)
    m, v = np.zeros_like(p), np.zeros_like(p)
    loss = net.train(idx, batch, 1e-3, want_loss=True)
    for s in range(steps):
        rows = idx[s * batch:(s + 1) * batch]
        step = engine.Mlp(p.astype(np.float32))
        g, one = step.gradient(X[rows], T[rows])
        step.close()
        assert abs(one - loss[s]) <= 1e-4 * abs(one)
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g.astype(np.float64) ** 2
        p = p - 1e-3 * (m / (1 - 0.9 ** (s + 1))) / (np.sqrt(v / (1 - 0.999 ** (s + 1))) + 1e-8)
    # a step moves a weight by up to 1e-3; FP32 master weights, and the sign of
    # a gradient near zero may follow the order of its sum
    d = np.abs(net.params() - p)
    assert np.sqrt((d ** 2).mean()) <= 2e-5 * steps
    net.close()
