"""The order of the low-rank (-A) path's sums follows from N alone: rows in
blocks of 256 lanes, at most 512 blocks (lane t of block b: rows 256 b + t,
+ 256 blocks, ...), a wave's 64 lanes as a tree 32, 16, .. 1, the four waves in
order; the blocks' partials by lane t adding partials t and t + 256, then the
same trees.  The error norm feeds the step size, so another order is another
sequence of steps a few attempts later."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _wave_tree(v):
    """Sums of the last axis in stretches of 64: x[l] + x[l + 32], + 16, .. 1."""
    v = v.reshape(v.shape[:-1] + (-1, 64))
    n = 64
    while n > 1:
        n //= 2
        v = v[..., :n] + v[..., n:2 * n]
    return v[..., 0]


def _waves_in_order(v):
    """256 lanes: wave trees, then ((w0 + w1) + w2) + w3."""
    w = _wave_tree(v)
    return ((w[..., 0] + w[..., 1]) + w[..., 2]) + w[..., 3]


def _ordered_sum(x):
    """sum x_i in the documented order (columns separately)."""
    N = x.shape[0]
    blocks = min(-(-N // 256), 512)
    per = -(-N // (256 * blocks))
    lanes = np.zeros((per * blocks * 256,) + x.shape[1:], x.dtype)
    lanes[:N] = x
    lanes = lanes.reshape((per, blocks, 256) + x.shape[1:])
    acc = lanes[0]
    for p in range(1, per):
        acc = lanes[p] + acc
    part = np.zeros((512,) + x.shape[1:], x.dtype)
    part[:blocks] = _waves_in_order(np.moveaxis(acc, 1, -1))
    return _waves_in_order(np.moveaxis(part[:256] + part[256:], 0, -1))


@pytest.mark.parametrize("N", [65, 257, 9000, 16385, 65536, 65537, 100000, 131072, 131073, 150001, 300007])
@pytest.mark.parametrize("K", [1, 5, 9])
def test_sums_follow_n_alone(km, N, K):
    """theta = 0 (cos 1, sin 0) and one nonzero factor per row, in column
    i mod K: G_m = w_m sum X_im and C_i = X_im G_m need one rounding per
    addition and product, so NumPy gives their bits."""
    rng = np.random.default_rng(N + K)
    v = rng.standard_normal(N)
    X = np.zeros((N, K))
    col = np.arange(N) % K
    X[np.arange(N), col] = v
    w = rng.standard_normal(K)
    print(f"case lowrank order N={N} K={K}", flush=True)
    with km.Integrator(N, km.F64, atol=1e-9, c1=3.0) as it:
        it.set_omega(np.zeros(N))
        it.set_factor(X, w)
        it.use_factored("contract")
        _, cpl = it.rhs(np.zeros(N), couplings=True)
    G = _ordered_sum(X) * w
    C, S = np.asarray(cpl).reshape(N, 2).T
    assert np.array_equal(C, v * G[col])
    assert not S.any()


def _uncoupled_run(km, N, K, fixed, atol, h):
    """Zero weights: f = omega exactly on every path."""
    rng = np.random.default_rng(N)
    om = rng.standard_normal(N)
    th = 3.0 * rng.standard_normal(N)
    with km.Integrator(N, km.F64, atol=atol, c1=3.0, fixed=fixed) as it:
        it.set_omega(om)
        it.set_factor(rng.standard_normal((N, K)), np.zeros(K))
        it.use_factored("contract")
        it.set_state(th, 0.0, h)
        it.begin(h * np.arange(1, 8), 1.0, keep_rows=True, ring_rows=16)
        st = it.advance(6)
        times, hs = it.read_times()
        rows, r = it.read_outputs()
        y, t, hn = it.get_state()
    return {"accepted": st.accepted, "rejected": st.rejected, "times": times, "hs": hs, "rows": rows, "r": r, "y": y,
            "t": t, "h": hn}


@pytest.mark.parametrize("N,fixed", [(65, False), (257, False), (9000, False), (65537, False), (131072, False),
                                     (131073, True), (200000, True), (300007, True)])
@pytest.mark.parametrize("K", [5, 12])
def test_error_norm_and_order_parameter_groups(km, N, K, fixed):
    """The ranks above 16 take one launch per step of the product, its error
    partials and output rows per 256 consecutive rows; up to 131072 rows the
    fused launches have the same groups (past it with a fixed step: the output
    rows only).  Uncoupled oscillators leave rounding errors as the embedded
    error, which atol = 1e-19 turns into norms of order 1: h then carries every
    bit of the norm's sum."""
    print(f"case lowrank groups N={N} K={K} fixed={fixed}", flush=True)
    a = _uncoupled_run(km, N, K, fixed, 1e-19, 2.0 ** -6)
    b = _uncoupled_run(km, N, 17, fixed, 1e-19, 2.0 ** -6)
    assert a["accepted"] + a["rejected"] == 6
    for key in a:
        assert np.array_equal(a[key], b[key]), key
