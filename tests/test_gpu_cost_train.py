"""Training the cost model over several steps and epochs, parameter by
parameter against a float64 replay of the same Adam steps (mlp_ref's gradient
and the epochs' shuffles): the update that the next step's launch applies, the
one that has a launch of its own (beyond 32 blocks of 64 samples), and epochs
whose last batch is on the other side of that line."""
import numpy as np
import pytest

import mlp_ref
from rdmce_amd.learned import CostModel

pytestmark = pytest.mark.gpu

U = 2.0 ** -24  # unit roundoff of float32
M64 = (1 << 64) - 1
NT, F, H1, H2 = mlp_ref.NTRAIN, mlp_ref.F, mlp_ref.H1, mlp_ref.H2


def mix(x):
    z = (x + 0x9E3779B97F4A7C15) & M64
    z = ((z ^ (z >> 30)) * 0xBF58476D1CE4E5B9) & M64
    z = ((z ^ (z >> 27)) * 0x94D049BB133111EB) & M64
    return z ^ (z >> 31)


def shuffle(n, seed, epoch):
    """The epoch's order: Fisher-Yates from the top, xoshiro256** seeded by
    splitmix64, bounded numbers by multiply-shift."""
    state = mix(seed ^ mix((epoch + 0x632BE59BD9B4E019) & M64))
    s = [mix((state + k * 0x9E3779B97F4A7C15) & M64) for k in range(4)]

    def rotl(v, k):
        return ((v << k) | (v >> (64 - k))) & M64

    def number():
        r = (rotl((s[1] * 5) & M64, 7) * 9) & M64
        t = (s[1] << 17) & M64
        s[2] ^= s[0]
        s[3] ^= s[1]
        s[1] ^= s[2]
        s[0] ^= s[3]
        s[2] ^= t
        s[3] = rotl(s[3], 45)
        return r

    idx = np.arange(n)
    for i in range(n - 1, 0, -1):
        while True:
            m = number() * (i + 1)
            if (m & M64) >= i + 1 or (m & M64) >= ((1 << 64) - (i + 1)) % (i + 1):
                break
        j = m >> 64
        idx[i], idx[j] = idx[j], idx[i]
    return idx


def problem(n, seed):
    """Samples and weights whose ReLUs stay on their side: every
    pre-activation keeps away from 0, whatever the rounding."""
    rng = np.random.default_rng(seed)
    x = rng.uniform(-1, 1, (n, F)).astype(np.float32)
    y = rng.uniform(-1, 1, n).astype(np.float32)
    on1, on2 = np.where(np.arange(H1) % 4 < 3, 1.0, -1.0), np.where(np.arange(H2) % 4 < 3, 1.0, -1.0)
    p = np.concatenate([
        rng.uniform(-0.05, 0.05, F * H1), on1 * rng.uniform(0.8, 1.2, H1),
        rng.uniform(-0.02, 0.02, H1 * H2), on2 * rng.uniform(1.6, 2.0, H2),
        rng.uniform(-0.4, 0.4, H2), [0.1], rng.uniform(-0.1, 0.1, F), rng.uniform(0.8, 1.2, F)]).astype(np.float32)
    return x, y, p


def replay(p0, x, y, epochs, batch, lr, seed, rng=None):
    """Parameters and last epoch's mean loss in float64.  With `rng`, every
    value that float32 rounds is moved by up to its worst-case error: sums of
    k terms by k roundings of the sum of absolute values."""
    p = p0.astype(np.float64)
    b1, b2, eps, lr = (float(np.float32(v)) for v in (0.9, 0.999, 1e-8, lr))
    m, v = np.zeros(NT), np.zeros(NT)
    x, y = x.astype(np.float64), y.astype(np.float64)

    def err(shape=None):
        return 0.0 if rng is None else U * rng.uniform(-1, 1, shape)

    step, away = 0, np.inf
    for ep in range(epochs):
        order, loss = shuffle(len(y), seed, ep), 0.0
        for at in range(0, len(y), batch):
            rows = order[at:at + batch]
            xb, yb, cnt = x[rows], y[rows], len(rows)
            W1, c1, W2, c2, W3, c3, mean, istd = mlp_ref.unpack(p)
            xn = (xb - mean) * istd
            xn = xn + 2 * (np.abs(xb) + np.abs(mean)) * istd * err(xn.shape)
            z1 = xn @ W1 + c1
            z1 = z1 + (F + 1) * (np.abs(xn) @ np.abs(W1) + np.abs(c1)) * err(z1.shape)
            h1 = np.maximum(z1, 0)
            z2 = h1 @ W2 + c2
            z2 = z2 + (H1 + 1) * (h1 @ np.abs(W2) + np.abs(c2)) * err(z2.shape)
            h2 = np.maximum(z2, 0)
            out = h2 @ W3 + c3
            out = out + (H2 + 1) * (h2 @ np.abs(W3) + np.abs(c3)) * err(out.shape)
            away = min(away, np.abs(z1).min(), np.abs(z2).min())
            d = out - yb
            loss += float(d @ d)
            dy = 2 * d / cnt
            dy = dy + 3 * (np.abs(out) + np.abs(yb)) * 2 / cnt * err(dy.shape)
            d2 = np.outer(dy, W3) * (h2 > 0)
            d1 = d2 @ W2.T
            d1 = (d1 + (H2 + 1) * (np.abs(d2) @ np.abs(W2.T)) * err(d1.shape)) * (h1 > 0)
            k = 64 + -(-cnt // 64)

            def entry(a, b):
                s = a.T @ b
                return (s + k * (np.abs(a).T @ np.abs(b)) * err(s.shape)).ravel()

            one = np.ones((cnt, 1))
            g = np.concatenate([entry(xn, d1), entry(one, d1), entry(h1, d2), entry(one, d2), entry(h2, dy[:, None]),
                                entry(one, dy[:, None])])
            step += 1
            m = (b1 * m + (1 - b1) * g) * (1 + 2 * err(NT))
            v = (b2 * v + (1 - b2) * g * g) * (1 + 3 * err(NT))
            bc1, bc2 = 1 - b1 ** step, 1 - b2 ** step
            bc1, bc2 = bc1 + 2 * err(), bc2 + 2 * err()
            p[:NT] -= lr * (m / bc1) / (np.sqrt(v / bc2) + eps) * (1 + 4 * err(NT))
            p[:NT] *= 1 + err(NT)
    return p, loss / len(y), away


def tolerance(p0, x, y, epochs, batch, lr, seed, ref, loss):
    """What rounding can do: 8 times the largest deviation, entry by entry, of
    16 replays with worst-case errors of random sign.  (An update that used the
    wrong buffer, batch or step number is off by a good part of lr.)"""
    rng = np.random.default_rng(12345)
    tol, ltol = np.zeros(len(ref)), 0.0
    for _ in range(16):
        q, ql, _ = replay(p0, x, y, epochs, batch, lr, seed, rng)
        tol, ltol = np.maximum(tol, np.abs(q - ref)), max(ltol, abs(ql - loss))
    return 8 * tol, 8 * ltol + 1e-6 * loss


CASES = [(65, 64, 3), (130, 65, 2), (200, 8, 2), (100, 1000, 4),
         (2048, 2048, 3),   # 32 blocks: the next step applies the update
         (2049, 2049, 3),   # 33: a launch of its own
         (4500, 2112, 2),   # 33, 33 and 5 blocks, twice
         (2500, 2048, 2)]   # 32 and 8


@pytest.mark.parametrize("n,batch,epochs", CASES)
def test_training_follows_float64(n, batch, epochs):
    print(f"[gpu-case] cost training n={n} batch={batch} epochs={epochs}", flush=True)
    lr, seed = 1e-3, 17
    x, y, p0 = problem(n, n + batch)
    ref, loss, away = replay(p0, x, y, epochs, batch, lr, seed)
    assert away > 0.05  # no ReLU near its corner
    tol, ltol = tolerance(p0, x, y, epochs, batch, lr, seed, ref, loss)
    assert np.mean(tol[:NT] < 0.05 * lr) > 0.99
    m = CostModel(0)
    m.set_params(p0)
    got_loss = m.train(x, y, epochs=epochs, batch=batch, lr=lr, seed=seed)
    got = m.params().astype(np.float64)
    off = np.abs(got - ref) > tol
    assert not off.any(), (int(off.sum()), float(np.abs(got - ref).max()), float(tol[off].max()))
    assert abs(got_loss - loss) <= ltol
