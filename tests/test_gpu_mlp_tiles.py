"""rp_mlp_loss_grad at the edges of its tiles of 64 samples and 128 partial
rows, against numpy in 64 bits.

Tolerance: FP32 sums of up to n products (error at most about sqrt(n) eps32
of the sum of magnitudes, which is bounded by the largest gradient entry of a
weight whose inputs do not cancel) through two layers of 64: 1e-5 of the
largest entry covers n = 8300."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NP = 5122


def _reference(p, X, T, W):
    w1, b1 = p[:768].reshape(64, 12), p[768:832]
    w2, b2 = p[832:4928].reshape(64, 64), p[4928:4992]
    w3, b3 = p[4992:5120].reshape(2, 64), p[5120:]
    h1 = np.tanh(X @ w1.T + b1)
    h2 = np.tanh(h1 @ w2.T + b2)
    e = h2 @ w3.T + b3 - T
    dy = 2 * W * e / len(X)
    dz2 = (dy @ w3) * (1 - h2 * h2)
    dz1 = (dz2 @ w2) * (1 - h1 * h1)
    g = [dz1.T @ X, dz1.sum(0), dz2.T @ h1, dz2.sum(0), dy.T @ h2, dy.sum(0)]
    return (W * e * e).sum() / len(X), np.concatenate([a.ravel() for a in g])


@pytest.mark.parametrize("n", [1, 15, 16, 63, 64, 65, 8192, 8193, 8300])
def test_loss_grad_tiles(gpu, n):
    rng = np.random.default_rng(n)
    p = rng.normal(0, 0.3, NP).astype(np.float32)
    X = rng.normal(0, 1, (n, 12)).astype(np.float32)
    T = rng.normal(0, 1, (n, 2)).astype(np.float32)
    W = rng.uniform(0, 1, (n, 2)).astype(np.float32)
    loss, grad = _reference(*[a.astype(np.float64) for a in (p, X, T, W)])
    g = gpu.DeviceArray(np.full(NP, np.nan, np.float32))
    d = [gpu.DeviceArray(a) for a in (p, X, T, W)]
    for _ in range(2):
        assert gpu.mlp_loss_grad(*d, g) == pytest.approx(loss, rel=1e-5)
        assert np.abs(g.get() - grad).max() <= 1e-5 * np.abs(grad).max()
