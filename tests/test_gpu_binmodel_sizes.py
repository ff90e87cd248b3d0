"""The capacity model's forward pass and loss gradient at the edges of the
kernels' rounds (16-sample operand blocks, 32-sample rounds, 256 workgroups)
against float64 numpy.

Samples whose ReLU inputs or residual lie within 1e-3 of a kink are left out,
so both sides take the same branches.  Tolerances: every value is a sum of
products in binary32 (u = 2^-24); a chain of k operations is within k u of the
exact value relative to the sum of its terms' magnitudes, and the chains here
are at most F + H + H + 8 operations deep per sample, then at most
ceil(n / (32 * 256)) * 32 + 256 additions over the samples and workgroups."""
import numpy as np
import pytest

import rast as R

pytestmark = pytest.mark.gpu

F = 8
U = 2.0 ** -24


@pytest.fixture(scope="module")
def renderer():
    r = R.Renderer(64, 64)
    yield r
    r.close()


def layers(p, H):
    p = p.astype(np.float64)
    W1, b1, p = p[:F * H].reshape(H, F), p[F * H:F * H + H], p[F * H + H:]
    return W1, b1, p[:H * H].reshape(H, H), p[H * H:H * H + H], p[H * H + H:H * H + 2 * H], p[-1]


def samples(H, n, seed):
    """n samples away from every kink, and the parameters."""
    rng = np.random.default_rng(seed)
    p = rng.normal(0, 0.3, F * H + H + H * H + H + H + 1).astype(np.float32)
    W1, b1, W2, b2, W3, b3 = layers(p, H)
    xs, ys = [], []
    have = 0
    while have < n:
        x = rng.normal(0, 1, (2 * (n - have) + 64, F)).astype(np.float32)
        y = rng.normal(2, 1, x.shape[0]).astype(np.float32)
        a1 = x @ W1.T + b1
        a2 = np.maximum(a1, 0) @ W2.T + b2
        r = y - (np.maximum(a2, 0) @ W3 + b3)
        ok = (np.abs(a1).min(1) > 1e-3) & (np.abs(a2).min(1) > 1e-3) & (np.abs(r) > 1e-3)
        xs.append(x[ok])
        ys.append(y[ok])
        have += int(ok.sum())
    return p, np.concatenate(xs)[:n], np.concatenate(ys)[:n]


@pytest.mark.parametrize("hidden", [16, 32, 64])
@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 64, 65, 4099])
def test_forward_sizes(renderer, hidden, n):
    p, x, _ = samples(hidden, n, 100 * hidden + n)
    W1, b1, W2, b2, W3, b3 = layers(p, hidden)
    h1 = np.maximum(x @ W1.T + b1, 0)
    h2 = np.maximum(h1 @ W2.T + b2, 0)
    want = h2 @ W3 + b3
    mag = (((np.abs(x) @ np.abs(W1).T + np.abs(b1)) @ np.abs(W2).T + np.abs(b2)) @ np.abs(W3)) + abs(b3)
    m = R.BinModel(renderer, hidden=hidden, seed=3)
    m.set_params(p)
    got = m.forward(x)
    m.close()
    assert np.all(np.abs(got - want) <= (F + 2 * hidden + 8) * U * mag)


@pytest.mark.parametrize("hidden,n", [(h, n) for h in (16, 32, 64) for n in (1, 15, 17, 31, 32, 33, 1000, 8191, 8193)]
                         + [(64, 65536)])
def test_loss_gradient_sizes(renderer, hidden, n):
    tau = 0.9
    p, x, y = samples(hidden, n, 200 * hidden + n)
    W1, b1, W2, b2, W3, b3 = layers(p, hidden)
    x64 = x.astype(np.float64)

    def grads(a):
        """The gradient with signed terms (a = identity) or term magnitudes (a = abs)."""
        h1 = np.maximum(x64 @ W1.T + b1, 0)
        h2 = np.maximum(h1 @ W2.T + b2, 0)
        r = y - (h2 @ W3 + b3)
        g = a(np.where(r > 0, -tau, 1 - tau) / n)
        if a is np.abs:  # magnitudes through the layers
            m1 = (h1 > 0) * (np.abs(x64) @ np.abs(W1).T + np.abs(b1))
            m2 = (h2 > 0) * (m1 @ np.abs(W2).T + np.abs(b2))
        else:
            m1, m2 = h1, h2
        d2 = (h2 > 0) * (g[:, None] * a(W3))
        d1 = (h1 > 0) * (d2 @ a(W2))
        return np.concatenate([(d1.T @ a(x64)).ravel(), d1.sum(0), (d2.T @ m1).ravel(), d2.sum(0), m2.T @ g, [g.sum()]])

    want, mag = grads(lambda v: v), grads(np.abs)
    h2 = np.maximum(np.maximum(x64 @ W1.T + b1, 0) @ W2.T + b2, 0)
    r = y - (h2 @ W3 + b3)
    want_loss = np.where(r > 0, tau * r, (tau - 1) * r).mean()
    m = R.BinModel(renderer, hidden=hidden, seed=3)
    m.set_params(p)
    loss, got = m.loss_grad(x, y, tau)
    m.close()
    depth = F + 2 * hidden + 8 + -(-n // (32 * 256)) * 32 + 256
    assert np.all(np.abs(got - want) <= depth * U * mag + 1e-30)
    # a residual's rounding is bounded by its terms' magnitudes, at most their largest sum per sample
    mag_r = (((np.abs(x64) @ np.abs(W1).T + np.abs(b1)) @ np.abs(W2).T + np.abs(b2)) @ np.abs(W3)) + abs(b3) + np.abs(y)
    assert abs(loss - want_loss) <= depth * U * mag_r.mean()
