"""The cost model's training step at the edges of its blocks (64 samples) and
on both sides of the size where a step's update gets a launch of its own (32
blocks), against float64 NumPy."""
import numpy as np
import pytest

from rdmce_amd.learned import CostModel

pytestmark = pytest.mark.gpu

U = 2.0 ** -24  # unit roundoff of float32
SIZES = [8 * 32, 32, 32 * 32, 32, 32, 1, 8, 8]


def split(p):
    w1, b1, w2, b2, w3, b3, mean, istd = np.split(p, np.cumsum(SIZES)[:-1])
    return w1.reshape(8, 32), b1, w2.reshape(32, 32), b2, w3, b3, mean, istd


def forward(p, x):
    w1, b1, w2, b2, w3, b3, mean, istd = split(p)
    xn = (x - mean) * istd
    z1 = xn @ w1 + b1
    h1 = np.maximum(z1, 0)
    z2 = h1 @ w2 + b2
    h2 = np.maximum(z2, 0)
    return xn, z1, h1, z2, h2, h2 @ w3 + b3[0]


def gradient(p, x, y):
    """Gradient, loss, and the same sums over absolute values."""
    xn, z1, h1, z2, h2, out = forward(p, x)
    w2, w3 = split(p)[2], split(p)[4]
    d = out - y
    dy = 2 * d / len(y)

    def back(dy, w2, w3, xn, h1, h2):
        d2 = np.where(h2 > 0, dy[:, None] * w3, 0)
        d1 = np.where(h1 > 0, d2 @ w2.T, 0)
        return np.concatenate([(xn.T @ d1).ravel(), d1.sum(0), (h1.T @ d2).ravel(), d2.sum(0), h2.T @ dy, [dy.sum()]])

    # absolute values of every term, the forward sums' included
    w1, b1, _, b2, _, b3, _, _ = (np.abs(v) for v in split(p))
    axn = np.abs(xn)
    a1 = np.where(h1 > 0, axn @ w1 + b1, 0)
    a2 = np.where(h2 > 0, a1 @ np.abs(w2) + b2, 0)
    ady = 2 * (a2 @ np.abs(w3) + b3[0] + np.abs(y)) / len(y)
    return (back(dy, w2, w3, xn, h1, h2), (d * d).mean(), back(ady, np.abs(w2), np.abs(w3), axn, a1, a2),
            min(np.abs(z1).min(), np.abs(z2).min()))


def samples(n, seed):
    """Samples whose pre-activations keep away from 0 (a ReLU's side must not
    depend on the rounding)."""
    rng = np.random.default_rng(seed)
    m = CostModel(seed)
    m.fit_normalizer(rng.standard_normal((256, 8)).astype(np.float32))
    p = m.params().astype(np.float64)
    x = rng.standard_normal((4 * n + 64, 8)).astype(np.float32)
    _, z1, _, z2, _, _ = forward(p, x.astype(np.float64))
    keep = (np.abs(z1).min(1) > 2e-5) & (np.abs(z2).min(1) > 2e-5)
    x = np.ascontiguousarray(x[keep][:n])
    assert len(x) == n
    return m, x, rng.standard_normal(n).astype(np.float32)


@pytest.mark.parametrize("n", [1, 63, 64, 65, 1000, 2048, 2049, 5000])
def test_gradient_at_block_edges(n):
    print(f"[gpu-case] cost gradient n={n}", flush=True)
    m, x, y = samples(n, n)
    g, loss = m.gradient(x, y)
    ref, lref, absum, away = gradient(m.params().astype(np.float64), x.astype(np.float64), y.astype(np.float64))
    assert away > 1e-5
    blocks = -(-n // 64)
    k = 64 + blocks + 8 + 32 + 32 + 32 + 16  # roundings on the way to an entry
    assert np.all(np.abs(g - ref) <= k * U * absum + 1e-30)
    assert abs(loss - lref) <= 1e-4 * lref


@pytest.mark.parametrize("n,batch", [(1, 1), (65, 64), (130, 65), (2048, 2048), (2049, 2049), (4500, 2112)])
def test_one_epoch_is_gradient_steps(n, batch):
    """An epoch without a shuffle to speak of is Adam steps over its batches:
    with one batch an epoch, parameters after two epochs follow from two
    gradients (the first step moves each parameter by lr * sign(g))."""
    print(f"[gpu-case] cost train n={n} batch={batch}", flush=True)
    m, x, y = samples(n, n + 7)
    p0 = m.params().astype(np.float64)
    a = m.train(x, y, epochs=1, batch=batch, lr=1e-3, seed=3)
    p1 = m.params()
    m.set_params(p0.astype(np.float32))
    b = m.train(x, y, epochs=1, batch=batch, lr=1e-3, seed=3)
    assert a == b and np.array_equal(p1, m.params())  # deterministic
    assert np.array_equal(p1[-16:], p0[-16:].astype(np.float32))  # normalisation kept
    if batch >= n:
        g, lref, absum, _ = gradient(p0, x.astype(np.float64), y.astype(np.float64))
        k = 64 + 36 + 130
        sure = np.abs(g) > 1e3 * (k * U * absum + 1e-8)  # Adam's first step: lr * g / (|g| + eps)
        assert sure.any()
        step = p0[:-16] - p1[:-16]
        assert np.allclose(step[sure], 1e-3 * np.sign(g[sure]), rtol=5e-3, atol=1e-7)
        assert abs(a - lref) <= 1e-4 * lref
