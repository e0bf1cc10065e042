"""The matrix-unit training kernel (32 hidden units) against a float32 model
of its arithmetic on the host: minibatches of one sample, of whole and of
partial 16-sample blocks and 256-sample chunks, and a left-over of the data."""
import numpy as np
import pytest

from galp_amd import _abi

pytestmark = pytest.mark.gpu
H = 32


def shuffle(n, seed):
    """The library's seeded Fisher-Yates order."""
    m = (1 << 64) - 1
    order, s = list(range(n)), seed ^ 0x5DEECE66D
    for i in range(n - 1, 0, -1):
        s = (s + 0x9E3779B97F4A7C15) & m
        z = ((s ^ (s >> 30)) * 0xBF58476D1CE4E5B9) & m
        z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & m
        j = (z ^ (z >> 31)) % (i + 1)
        order[i], order[j] = order[j], order[i]
    return order


def train_host(p, x, y, epochs, batch, lr, seed):
    """Adam over the shuffled minibatches in float64."""
    n = len(x)
    order = shuffle(n, seed)
    x, y = x[order].astype(np.float64), y[order].astype(np.float64)
    p, b = p.astype(np.float64), min(batch, n)
    at = np.cumsum([4 * H, H, H * H, H, H])
    m, v, t = np.zeros_like(p), np.zeros_like(p), 0
    for _ in range(epochs):
        for o in range(0, n - b + 1, b):
            w1, b1, w2, b2, w3, b3 = np.split(p, at)
            w1, w2 = w1.reshape(H, 4), w2.reshape(H, H)
            xs = x[o:o + b]
            h1 = np.maximum(xs @ w1.T + b1, 0)
            z2 = h1 @ w2.T + b2
            g = (np.maximum(z2, 0) @ w3 + b3[0] - y[o:o + b]) / b
            d2 = np.where(z2 > 0, g[:, None] * w3, 0)
            d1 = np.where(h1 > 0, d2 @ w2, 0)
            grad = np.concatenate([(d1.T @ xs).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0),
                                   np.maximum(z2, 0).T @ g, [g.sum()]])
            t += 1
            m, v = 0.9 * m + 0.1 * grad, 0.999 * v + 0.001 * grad * grad
            p = p - lr * (m / (1 - 0.9 ** t)) / (np.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
    return p


@pytest.mark.parametrize("n,batch,epochs", [(1, 1, 2), (15, 15, 2), (33, 16, 2), (300, 255, 3), (600, 256, 2),
                                            (1000, 257, 2), (1300, 512, 2), (777, 2000, 3)])
def test_train_matches_host(ctx, n, batch, epochs):
    print(f"[train] n={n} batch={batch} epochs={epochs}", flush=True)
    rng = np.random.default_rng(n)
    x = rng.uniform(-1, 14, size=(n, 4)).astype(np.float32)
    y = (0.5 * x[:, 0] + 0.1 * x[:, 3] + 1).astype(np.float32)
    p0 = _abi.mlp_init(H, n)
    got, _ = _abi.mlp_train(ctx, H, p0, x, y, epochs=epochs, batch=batch, lr=1e-3, seed=3)
    want = train_host(p0, x, y, epochs, batch, 1e-3, 3)
    # Adam steps of at most lr * (1 + small) each: a sign of a
    # near-zero gradient may differ in single precision, which moves a
    # parameter by up to 2 lr a step; anything but a few such parameters is
    # within float32's accumulation error of a step
    steps = epochs * (n // min(batch, n))
    off = np.abs(got - want)
    assert off.max() <= 2.2e-3 * steps
    assert np.mean(off > 1e-5 * steps) < 0.05
