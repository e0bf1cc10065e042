"""The size and sign of every gradient the matrix-unit training kernel (32
hidden units) forms, block by block of the parameter vector.

Adam's first step moves a parameter by lr * g / (|g| + 1e-8), which shows g
itself only where it is about as small as 1e-8.  So the networks here have one
layer scaled down to S (and its bias, and the targets): "w3" makes the
gradients of W3 and b3 of the order of S, "w2" those of W2, b2 and b3, "w1"
those of W1, b1, b2 and b3.  One minibatch, one step, against float64; the
tolerance is the float32 rounding of the sums, carried through layer by layer
in first order (units of 2^-24, any order of summation), and it is required to
be far below the steps, so that a block of wrong gradients cannot pass."""
import numpy as np
import pytest

from galp_amd import _abi
from test_gpu_training import shuffle

H, S, EPS, LR, U = 32, 2e-8, 1e-8, 1e-2, 2.0 ** -24
BLOCKS = ("w1", "b1", "w2", "b2", "w3", "b3")
AT = np.cumsum([4 * H, H, H * H, H, H])
SHOWN = {"w3": ("w3", "b3"), "w2": ("w2", "b2", "b3"), "w1": ("w1", "b1", "b2", "b3")}


def network(layer, rng):
    w = {"w1": rng.uniform(-0.5, 0.5, (H, 4)), "b1": rng.uniform(-0.5, 0.5, H),
         "w2": rng.uniform(-0.3, 0.3, (H, H)), "b2": rng.uniform(-0.3, 0.3, H),
         "w3": rng.uniform(-0.5, 0.5, H), "b3": rng.uniform(-0.5, 0.5, 1)}
    for b in SHOWN[layer]:
        w[b] = w[b] * S
    return np.concatenate([w[b].ravel() for b in BLOCKS]).astype(np.float32)


def split(p):
    w1, b1, w2, b2, w3, b3 = np.split(p.astype(np.float64), AT)
    return w1.reshape(H, 4), b1, w2.reshape(H, H), b2, w3, b3


def forward(p, x):
    """z1, z2 and the output in float64, each with its rounding bound."""
    w1, b1, w2, b2, w3, b3 = split(p)
    z1, e1 = x @ w1.T + b1, 5 * U * (np.abs(x) @ np.abs(w1).T + np.abs(b1))
    h1 = np.maximum(z1, 0)
    z2 = h1 @ w2.T + b2
    e2 = 34 * U * (h1 @ np.abs(w2).T + np.abs(b2)) + e1 @ np.abs(w2).T
    h2 = np.maximum(z2, 0)
    return z1, e1, z2, e2, h2 @ w3 + b3, 34 * U * (h2 @ np.abs(w3) + np.abs(b3)) + e2 @ np.abs(w3)


def samples(p, n, rng):
    """n samples whose hidden units are on either side of zero beyond doubt."""
    x = rng.uniform(-1, 14, size=(4 * n + 64, 4)).astype(np.float32)
    z1, e1, z2, e2, out, _ = forward(p, x.astype(np.float64))
    x = x[np.all(np.abs(z1) > 8 * e1, 1) & np.all(np.abs(z2) > 8 * e2, 1)][:n]
    assert len(x) == n
    return x, (S * rng.uniform(-30, 30, n)).astype(np.float32)


def one_step(p, x, y):
    """The parameters after one Adam step over (x, y), and the tolerance."""
    w1, b1, w2, b2, w3, b3 = split(p)
    x, y, n = x.astype(np.float64), y.astype(np.float64), len(x)
    z1, e1, z2, e2, out, eo = forward(p, x)
    h1, h2, on1, on2 = np.maximum(z1, 0), np.maximum(z2, 0), z1 > 0, z2 > 0
    g, eg = (out - y) / n, (eo + 3 * U * np.abs(out - y)) / n
    d2, f2 = on2 * np.outer(g, w3), on2 * np.outer(eg + U * np.abs(g), np.abs(w3))
    d1, f1 = on1 * (d2 @ w2), on1 * (f2 @ np.abs(w2) + 33 * U * (np.abs(d2) @ np.abs(w2)))
    k = (n + 1) * U   # a sum over the samples, in any order

    def outer(a, fa, b, fb):   # sum over the samples of a * b
        aa, bb = np.abs(a), np.abs(b)
        return a.T @ b, fa.T @ bb + aa.T @ fb + k * (aa.T @ bb)

    zero, one = np.zeros_like(x), np.ones((n, 1))
    parts = [outer(d1, f1, x, zero), outer(d1, f1, one, 0 * one), outer(d2, f2, h1, on1 * e1),
             outer(d2, f2, one, 0 * one), outer(h2, on2 * e2, g[:, None], eg[:, None]),
             outer(g[:, None], eg[:, None], one, 0 * one)]
    grad, err = (1.0 * np.concatenate([q[i].ravel() for q in parts]) for i in (0, 1))
    a = np.abs(grad)
    step = LR * grad / (a + EPS)
    tol = 1.01 * LR * EPS * err / (np.maximum(a - err, 0) + EPS) ** 2 + 16 * U * np.abs(step) + 2 * U * np.abs(p)
    return p.astype(np.float64) - step, tol, grad


SIZES = [(1, 1), (15, 15), (16, 16), (17, 17), (255, 255), (256, 256), (257, 257), (300, 256), (512, 512), (700, 600)]


def case(layer, n, batch):
    rng = np.random.default_rng([n, batch, BLOCKS.index(layer)])
    p = network(layer, rng)
    x, y = samples(p, n, rng)
    order = shuffle(n, 5)[:batch]   # the rest of the data is left over
    want, tol, grad = one_step(p, x[order], y[order])
    shown = np.concatenate([np.full(size, b in SHOWN[layer]) for b, size in zip(BLOCKS, np.diff([0, *AT, AT[-1] + 1]))])
    return p, x, y, want, tol, grad, shown


@pytest.mark.parametrize("layer", ["w1", "w2", "w3"])
@pytest.mark.parametrize("n,batch", SIZES)
def test_tolerance_tells_gradients_apart(layer, n, batch):
    """Gradients that are off by a twentieth, or have the other sign, are
    outside the tolerance in the blocks the case is for."""
    p, x, y, want, tol, grad, shown = case(layer, n, batch)
    grad, tol = grad[shown], tol[shown]
    used = np.abs(grad) > 1e-2 * EPS   # units that are off for all samples have none
    assert used.sum() >= 0.3 * shown.sum()

    def moved(g):
        return LR * g / (np.abs(g) + EPS)

    for wrong in (0 * grad, -grad, 1.05 * grad, 0.95 * grad):
        off = np.abs(moved(wrong) - moved(grad)) > tol
        assert off[used].mean() > 0.9


@pytest.mark.gpu
@pytest.mark.parametrize("layer", ["w1", "w2", "w3"])
@pytest.mark.parametrize("n,batch", SIZES)
def test_first_step(ctx, layer, n, batch):
    p, x, y, want, tol, _, _ = case(layer, n, batch)
    print(f"[train] {layer} n={n} batch={batch}", flush=True)
    got, _ = _abi.mlp_train(ctx, H, p, x, y, epochs=1, batch=batch, lr=LR, seed=5)
    off = np.abs(got.astype(np.float64) - want)
    for b, o, t in zip(BLOCKS, np.split(off, AT), np.split(tol, AT)):
        assert np.all(o <= t), (b, float((o / t).max()))
