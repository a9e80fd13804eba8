"""The network's fused path (hidden and inputs up to 256) at the edges of its
tiles: 16 rows per workgroup, weights padded to 64, batch slices of 12-row
steps, prediction chunks of 32768 rows; and the general path just beyond it.
Tolerances as in test_mlp.py (FP32 sums against FP64)."""
import numpy as np
import pytest

import mlp_ref
from test_mlp import _params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_in,hidden,B", [(1, 1, 1), (16, 64, 15), (17, 65, 16), (64, 128, 17), (65, 200, 1000),
                                           (256, 256, 33), (19, 192, 10007), (257, 64, 50), (19, 257, 50)])
def test_gradient_and_probabilities(tracker, n_in, hidden, B):
    from elegant_amd import learned
    m = learned.MLP(tracker, n_in=n_in, hidden=hidden, seed=3)
    p = _params(n_in, hidden, 6).astype(np.float32)
    rng = np.random.default_rng(B)
    X = rng.normal(size=(B, n_in)).astype(np.float32)
    y = (rng.random(B) < 0.4).astype(np.float32)
    for scale in (1.0, 0.5):  # parameters set twice: the tiled copies follow
        q = (p * np.float32(scale)).astype(np.float32)
        m.set_params(q)
        g, l = m.gradient(X, y)
        gr, lr = mlp_ref.gradient(q.astype(np.float64), X.astype(np.float64), y, n_in, hidden)
        assert abs(l - lr) < 1e-5 * max(1.0, abs(lr))
        for a, b in zip(mlp_ref.unpack(gr, n_in, hidden), mlp_ref.unpack(g, n_in, hidden)):
            assert np.linalg.norm(a - b) <= 2e-4 * np.linalg.norm(a) + 1e-9
        assert np.max(np.abs(m.predict(X) - mlp_ref.predict(q, X, n_in, hidden))) < 1e-5
    m.close()


@pytest.mark.parametrize("n", [1, 17, 8192, 8193, 32768, 32769, 98305])
def test_prediction_chunks(tracker, n):
    from elegant_amd import learned
    m = learned.MLP(tracker, hidden=100, seed=4)
    X = np.random.default_rng(n).normal(size=(n, 19)).astype(np.float32)
    ref = mlp_ref.predict(m.params(), X, 19, 100)
    for _ in range(2):
        assert np.max(np.abs(m.predict(X) - ref)) < 1e-5
    m.close()


def test_training_steps_match_adam(tracker):
    """six steps (two epochs of three batches) against Adam in 64 bits on the
    same order of samples; the same training twice gives the same bits"""
    from elegant_amd import learned
    n, B = 3 * 1000 + 17, 1000
    rng = np.random.default_rng(8)
    X = rng.normal(size=(n, 19)).astype(np.float32)
    y = (X[:, 0] ** 2 + X[:, 1] ** 2 < 1.0).astype(np.float32)
    runs = []
    for _ in range(2):
        m = learned.MLP(tracker, seed=5)
        w = m.params().astype(np.float64)
        losses = m.train(X, y, epochs=2, batch=B, lr=1e-3, seed=7)
        runs.append((m.params(), losses))
        m.close()
    assert np.array_equal(runs[0][0], runs[1][0]) and np.array_equal(runs[0][1], runs[1][1])

    class Mix:  # the library's SplitMix64 order
        s = 7

        def uni(self):
            self.s = (self.s + 0x9E3779B97F4A7C15) % 2 ** 64
            z = self.s
            z = (z ^ z >> 30) * 0xBF58476D1CE4E5B9 % 2 ** 64
            z = (z ^ z >> 27) * 0x94D049BB133111EB % 2 ** 64
            return ((z ^ z >> 31) >> 11) / 2 ** 53

    mix, mo, v, t, ref = Mix(), np.zeros_like(w), np.zeros_like(w), 0, []
    for _ in range(2):
        p = list(range(n))
        for i in range(n - 1, 0, -1):
            j = int(mix.uni() * (i + 1))
            p[i], p[j] = p[j], p[i]
        total = 0.0
        for b in range(n // B):
            rows = p[b * B:(b + 1) * B]
            g, l = mlp_ref.gradient(w, X[rows].astype(np.float64), y[rows])
            total += l
            t += 1
            mo = 0.9 * mo + 0.1 * g
            v = 0.999 * v + 0.001 * g * g
            w = w - 1e-3 * (mo / (1 - 0.9 ** t)) / (np.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
        ref.append(total / (n // B))
    assert np.allclose(runs[0][1], ref, rtol=1e-4)
    # a step moves each weight by up to 1e-3 whatever its gradient's size, so
    # rounding of the smallest gradients shows: a few 1e-4 of the norm
    assert np.linalg.norm(runs[0][0] - w) < 2e-3 * np.linalg.norm(w)


def _embedded(p, n_in, hidden, wide):
    """the parameters of the same net with inputs that nothing sends"""
    w = np.zeros((hidden, wide), np.float32)
    w[:, :n_in] = p[:hidden * n_in].reshape(hidden, n_in)
    return np.concatenate([w.ravel(), p[hidden * n_in:]])


def _without(p, n_in, hidden, wide):
    w = p[:hidden * wide].reshape(hidden, wide)
    assert not w[:, n_in:].any()
    return np.concatenate([w[:, :n_in].ravel(), p[hidden * wide:]])


@pytest.mark.parametrize("n_in,hidden,B", [(1, 1, 1), (19, 1, 63), (16, 15, 64), (19, 64, 65), (17, 65, 129),
                                           (33, 100, 250), (19, 129, 257), (19, 192, 831), (256, 256, 127),
                                           (19, 256, 831), (19, 100, 1000), (19, 64, 3000)])
def test_same_bits_as_the_general_path(tracker, n_in, hidden, B):
    """a net of 257 inputs takes the general path; with the inputs beyond n_in
    always zero it is the same net, and every sum has the same order wherever
    both cut the batch into as many slices (B below 64 times the general
    path's 256 / tiles of the first layer): the gradients, six Adam steps and
    the probabilities are equal bit for bit"""
    from elegant_amd import learned
    wide = 257
    assert B // 64 <= max(1, 256 // (-(-hidden // 64) * 5))
    rng = np.random.default_rng(B + hidden)
    X = rng.normal(size=(3 * B, n_in)).astype(np.float32)
    y = (rng.random(3 * B) < 0.4).astype(np.float32)
    XW = np.zeros((3 * B, wide), np.float32)
    XW[:, :n_in] = X
    a = learned.MLP(tracker, n_in=n_in, hidden=hidden, seed=3)
    b = learned.MLP(tracker, n_in=wide, hidden=hidden, seed=3)
    p = a.params()
    b.set_params(_embedded(p, n_in, hidden, wide))
    ga, la = a.gradient(X[:B], y[:B])
    gb, lb = b.gradient(XW[:B], y[:B])
    assert la == lb and np.array_equal(ga, _without(gb, n_in, hidden, wide))
    la = a.train(X, y, epochs=2, batch=B, lr=1e-3, seed=7)
    lb = b.train(XW, y, epochs=2, batch=B, lr=1e-3, seed=7)
    assert np.array_equal(la, lb) and np.array_equal(a.params(), _without(b.params(), n_in, hidden, wide))
    assert np.array_equal(a.predict(X), b.predict(XW))
    a.close()
    b.close()


@pytest.mark.parametrize("B", [4096, 10007])
def test_same_bits_beyond_the_first_layer(tracker, B):
    """larger batches, which the general net's first layer cuts differently:
    the other layers' gradients"""
    from elegant_amd import learned
    n_in, hidden, wide = 19, 256, 257
    rng = np.random.default_rng(B)
    X = rng.normal(size=(B, n_in)).astype(np.float32)
    y = (rng.random(B) < 0.4).astype(np.float32)
    XW = np.zeros((B, wide), np.float32)
    XW[:, :n_in] = X
    a = learned.MLP(tracker, n_in=n_in, hidden=hidden, seed=3)
    b = learned.MLP(tracker, n_in=wide, hidden=hidden, seed=3)
    b.set_params(_embedded(a.params(), n_in, hidden, wide))
    ga, la = a.gradient(X, y)
    gb, lb = b.gradient(XW, y)
    assert la == lb and np.array_equal(ga[hidden * n_in:], _without(gb, n_in, hidden, wide)[hidden * n_in:])
    a.close()
    b.close()
