"""The proposer's gradient and training kernels at the edges of their sample
batches (32 per register set, 64 per factor load), against the FP64 oracle
network on the same FP16-rounded weights."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _data(km, n, seed):
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((n, 8)).astype(np.float32)
    y = (0.3 * np.tanh(X[:, 0]) - 0.2 * X[:, 3] + 0.1 * X[:, 6] * X[:, 7]).astype(np.float32)
    return X, y, (0.15 * rng.standard_normal(km.proposer_param_count())).astype(np.float32)


@pytest.mark.parametrize("n", [1, 31, 32, 33, 63, 64, 65, 95, 97, 128, 1000])
def test_gradient_at_batch_edges(km, orc, n):
    """Each parameter is n sequential FP32 fmas of terms with a relative error
    of a few 2^-22 (tanhf, 64-term dot products in FP32): n 2^-24 + 2^-20 of
    the sum of the terms' magnitudes, below 1e-4 of the largest gradient
    times the terms' cancellation (at most ~4 here)."""
    X, y, w0 = _data(km, n, 11 + n)
    print(f"case mlp gradient n={n}", flush=True)
    with km.Mlp(w0) as m:
        _, w16 = m.weights()
        loss, g = m.loss_grad(X, y)
    lo, go, _ = orc.mlp_loss_grad(w16.astype(np.float64), X.astype(np.float64), y.astype(np.float64))
    assert abs(loss - lo) < 1e-5 * max(1.0, lo)
    assert np.max(np.abs(g - go)) < 2e-4 * np.abs(go).max()


@pytest.mark.parametrize("n,batch", [(130, 64), (97, 97), (97, 200), (66, 1)])
def test_epoch_equals_single_minibatches(km, n, batch):
    """One call over an epoch = one call per minibatch: the same weights bit
    for bit, and the epoch's loss is the samples' mean of the minibatches'."""
    X, y, w0 = _data(km, n, 5)
    print(f"case mlp epoch n={n} batch={batch}", flush=True)
    with km.Mlp(w0) as a, km.Mlp(w0) as b:
        hist = a.train(X, y, epochs=1, batch=batch, lr=1e-3)
        tot = 0.0
        for s in range(0, n, batch):
            k = min(batch, n - s)
            tot += k * b.train(X[s:s + batch], y[s:s + batch], epochs=1, batch=batch, lr=1e-3)[0]
        wa, wb = a.weights(), b.weights()
    assert np.array_equal(wa[0], wb[0]) and np.array_equal(wa[1], wb[1])
    assert abs(hist[0] - tot / n) <= 1e-12 * abs(hist[0])
