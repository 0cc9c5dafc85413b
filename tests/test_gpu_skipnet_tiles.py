"""The skip network's kernels at the edges of their workgroups (4 samples) and of the
samples that a gradient round holds (256): forward pass, loss and every gradient
against numpy in doubles, and bit for bit against numpy in FP32 with the same order.

Tolerance: each value is a chain of at most three FP32 contractions of at most 132
terms (hidden layers, deltas) and one over the batch, so it is off by at most
(3 * 132 + n + 16) 2^-24 times the same chain of absolute values, the bound used
(a hidden unit within that bound of 0 may fall on the other side of the ReLU:
rows with one are left out of the inputs)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _split(p):
    o = np.cumsum([64 * 132, 64, 64 * 64, 64, 64])
    w1, b1, w2, b2, w3, b3 = np.split(p, o)
    return w1.reshape(64, 132), b1, w2.reshape(64, 64), b2, w3, b3[0]


@pytest.mark.parametrize("n", [1, 2, 15, 16, 17, 64, 65, 127, 128, 129, 300])
def test_gradient_tiles(gpu, n):
    rng = np.random.default_rng(n)
    p = (rng.normal(size=gpu.SKIPNET_PARAMS) * 0.15).astype(np.float32)
    u = (3 * 132 + n + 16) * 2.0 ** -24
    w1, b1, w2, b2, w3, b3 = _split(p.astype(np.float64))

    def layers(xd):  # the layers before their ReLU, and the same chains of absolute values
        z1 = xd @ w1.T + b1
        z2 = np.maximum(z1, 0) @ w2.T + b2
        a1 = np.abs(xd) @ np.abs(w1).T + np.abs(b1)
        return z1, z2, a1, a1 @ np.abs(w2).T + np.abs(b2)

    x = rng.normal(size=(4 * n + 8, gpu.SKIPNET_INPUTS)).astype(np.float32)
    z1, z2, a1, a2 = layers(x.astype(np.float64))
    x = x[(np.abs(z1) > u * a1).all(1) & (np.abs(z2) > u * a2).all(1)][:n]
    assert len(x) == n
    t = rng.normal(size=n).astype(np.float32)
    net = gpu.SkipNet()
    net.set(p, np.zeros(gpu.SKIPNET_INPUTS, np.float32), np.ones(gpu.SKIPNET_INPUTS, np.float32))
    y = net.predict(x)
    loss, g = net.gradient(x, t)

    xd, td = x.astype(np.float64), t.astype(np.float64)
    z1, z2, a1, a2 = layers(xd)
    h1, h2 = np.maximum(z1, 0), np.maximum(z2, 0)
    yd, ya = h2 @ w3 + b3, a2 @ np.abs(w3) + np.abs(b3)
    dy, dya = 2 * (yd - td) / n, 2 * (ya + np.abs(td)) / n
    d2, d2a = np.outer(dy, w3) * (z2 > 0), np.outer(dya, np.abs(w3)) * (z2 > 0)
    d1, d1a = (d2 @ w2) * (z1 > 0), (d2a @ np.abs(w2)) * (z1 > 0)
    want = np.concatenate([(d1.T @ xd).ravel(), d1.sum(0), (d2.T @ h1).ravel(), d2.sum(0), h2.T @ dy, [dy.sum()]])
    top = np.concatenate([(d1a.T @ np.abs(xd)).ravel(), d1a.sum(0), (d2a.T @ a1).ravel(), d2a.sum(0), a2.T @ dya,
                          [dya.sum()]])
    assert (np.abs(y - yd) <= u * ya).all()
    assert (np.abs(g - want) <= u * top + 1e-37).all()
    assert abs(loss - np.mean((yd - td) ** 2)) <= u * np.mean((ya + np.abs(td)) ** 2)


@pytest.mark.parametrize("n", [1, 3, 4, 5, 31, 33, 255, 256, 257, 513])
def test_sums_keep_their_order(gpu, n):
    """Every sum one rounded term after the other, over the inputs and over the batch: no tolerance."""
    rng = np.random.default_rng(100 + n)
    p = (rng.normal(size=gpu.SKIPNET_PARAMS) * 0.15).astype(np.float32)
    x = rng.normal(size=(n, gpu.SKIPNET_INPUTS)).astype(np.float32)
    t = rng.normal(size=n).astype(np.float32)
    w1, b1, w2, b2, w3, b3 = _split(p)

    def chain(s, terms):
        for v in terms:
            s = s + v
        return s

    h1 = np.maximum(chain(np.tile(b1, (n, 1)), (w1[:, k] * x[:, k:k + 1] for k in range(132))), np.float32(0))
    h2 = np.maximum(chain(np.tile(b2, (n, 1)), (w2[:, k] * h1[:, k:k + 1] for k in range(64))), np.float32(0))
    y = chain(np.full(n, b3), (w3[k] * h2[:, k] for k in range(64)))
    dy = np.float32(2) * (y - t) / np.float32(n)
    d2 = np.where(h2 > 0, dy[:, None] * w3, np.float32(0))
    d1 = np.where(h1 > 0, chain(np.zeros_like(d2), (w2[i] * d2[:, i:i + 1] for i in range(64))), np.float32(0))

    def grad(d, h):
        return chain(np.zeros((d.shape[1], h.shape[1]), np.float32), (d[b][:, None] * h[b] for b in range(n))).ravel()

    one = np.ones((n, 1), np.float32)
    want = np.concatenate([grad(d1, x), grad(d1, one), grad(d2, h1), grad(d2, one), grad(dy[:, None], h2),
                           grad(dy[:, None], one)])
    net = gpu.SkipNet()
    net.set(p, np.zeros(gpu.SKIPNET_INPUTS, np.float32), np.ones(gpu.SKIPNET_INPUTS, np.float32))
    assert y.dtype == want.dtype == np.float32
    assert np.array_equal(net.predict(x), y)
    assert np.array_equal(net.gradient(x, t)[1], want)


@pytest.mark.parametrize("n,batch", [(5, 8), (33, 16), (300, 100)])
def test_training_repeats_bit_for_bit(gpu, n, batch):
    rng = np.random.default_rng(n)
    x = rng.normal(size=(n, gpu.SKIPNET_INPUTS)).astype(np.float32)
    t = rng.normal(size=n).astype(np.float32)
    net = gpu.SkipNet()
    runs = []
    for _ in range(2):
        curve = net.train(x, t, epochs=70, batch=batch, lr=2e-3, seed=3)
        runs.append((curve, net.get()[0]))
    assert np.array_equal(runs[0][0], runs[1][0]) and np.array_equal(runs[0][1], runs[1][1])
    assert np.isfinite(runs[0][0]).all() and runs[0][0][-1] < runs[0][0][0]
