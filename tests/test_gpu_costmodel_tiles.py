"""The cost model's matrix-core kernels at the edges of their tiles and
batches: sample counts around 16 (a wave's predictions), 64 (a step), the
pinned staging's capacity and one batch more than the gradient's workgroups,
against float64. FP32 sums of at most 64 terms a layer keep a prediction
within about 64 * 2^-24 of its terms' size: 1e-5 of the predictions' root
mean square covers the three layers; a gradient sums further over the
samples, 1e-5 of its root mean square was above every count measured."""
import numpy as np
import pytest

import av1ongpu_amd as pkg
from mlp_ref import init_params, loss_and_grad, predict_us, standardise

pytestmark = pytest.mark.gpu


def _model(seed, n):
    rng = np.random.default_rng(seed)
    p = init_params(rng).astype(np.float32)
    p[24 * 64:24 * 64 + 64] = rng.normal(0, 0.2, 64)
    p[-129 - 64:-129] = rng.normal(0, 0.2, 64)
    X = rng.gamma(1.5, 8.0, (n, pkg.CM_FEATURES)).astype(np.float32)
    y = (X[:, 0] + 0.2 * X[:, 1] * X[:, 2] + 3).astype(np.float32)
    mean, dev = X.mean(0) * np.float32(0.9), X.std(0) + np.float32(0.5)
    cm = pkg.CostModel(seed=1)
    cm.set_params(p)
    cm.set_norm(mean, dev, 20.0, 11.0)
    return cm, p, X, y, mean, dev


def _off(got, want):
    return np.abs(got - want).max() / np.sqrt(np.mean(np.square(want)))


@pytest.mark.parametrize("n", [1, 15, 16, 17, 63, 4096, 4097])
def test_predict(n):
    cm, p, X, _y, mean, dev = _model(n, n)
    assert _off(cm.predict(X), predict_us(p, X, mean, dev, 20.0, 11.0)) < 1e-5


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 129, 257 * 64 + 1])
def test_gradients(n):
    cm, p, X, y, mean, dev = _model(n, n)
    g, loss = cm.gradients(X, y)
    want_loss, want = loss_and_grad(p, *standardise(X, y, mean, dev, 20.0, 11.0))
    assert abs(loss - want_loss) <= 1e-5 * want_loss
    assert _off(g, want) < 1e-4 and np.linalg.norm(g - want) < 1e-5 * np.linalg.norm(want)


@pytest.mark.parametrize("n,epochs", [(2, 1), (37, 3), (64, 4)])
def test_train_one_batch(n, epochs):
    """With one batch an epoch the drawn order does not matter: the steps
    are Adam's on the mean gradient."""
    cm, p, X, y, mean, dev = _model(n, n)
    Xs, ys = standardise(X, y, mean, dev, 20.0, 11.0)
    losses = cm.train(X, y, epochs=epochs, lr=1e-3, seed=2, set_norm=False)
    w = p.astype(np.float64)
    m, v = np.zeros_like(w), np.zeros_like(w)
    for t in range(1, epochs + 1):
        loss, g = loss_and_grad(w, Xs, ys)
        assert abs(losses[t - 1] - loss) <= 1e-4 * loss
        m, v = 0.9 * m + 0.1 * g, 0.999 * v + 0.001 * g * g
        w = w - 1e-3 * (m / (1 - 0.9 ** t)) / (np.sqrt(v / (1 - 0.999 ** t)) + 1e-8)
    # a gradient near zero may round to either sign, and a step is then up to
    # a learning rate off; all but a few weights agree to rounding
    d = np.abs(cm.params() - w)
    assert np.median(d) < 1e-6 and (d > 1e-5).mean() < 0.02 and d.max() <= 2.1e-3 * epochs


def test_train_repeats():
    """The same samples, weights and seed train to the same bits: every sum,
    the loss's too, has one order."""
    runs = []
    for _ in range(3):
        cm, _p, X, y, _mean, _dev = _model(5, 4000)
        losses = cm.train(X, y, epochs=2, lr=1e-3, seed=3, set_norm=False)
        runs.append((list(losses), cm.params().tobytes()))
    assert runs[0] == runs[1] == runs[2]


def test_predict_again_and_from_threads():
    """Calls of one model share its staging: one after the other and from
    several threads, each gets its own samples' predictions."""
    from concurrent.futures import ThreadPoolExecutor
    cm, p, X, _y, mean, dev = _model(9, 4096)
    parts = [X[i * 300:i * 300 + n] for i, n in enumerate((300, 17, 1000, 64, 300, 2040))]
    want = [predict_us(p, x, mean, dev, 20.0, 11.0) for x in parts]
    for x, w in zip(parts + parts[::-1], want + want[::-1]):
        assert _off(cm.predict(x), w) < 1e-5
    with ThreadPoolExecutor(4) as pool:
        for got, w in zip(pool.map(cm.predict, parts * 20), want * 20):
            assert _off(got, w) < 1e-5
