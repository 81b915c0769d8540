"""The low-rank (-A) path where its launch shape changes: ranks on both sides
of the exact-rank kernels and of their thread bounds, sizes on both sides of a
wave, of 256 rows, of the widest workgroups and of one row per thread."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _problem(km, N, K, dtype, seed):
    rng = np.random.default_rng(seed)
    X = rng.standard_normal((N, K)).astype(dtype)
    w = np.full(K, -1.0 / (N * max(K, 1)), dtype)
    return rng.uniform(-3, 3, N).astype(dtype), rng.standard_normal(N).astype(dtype), X, w


def _field(theta, om, X, w, c1):
    th, x = theta.astype(np.float64), X.astype(np.float64)
    G = w.astype(np.float64)[:, None] * (x.T @ np.stack([np.cos(th), np.sin(th)], 1))
    C = x @ G
    return om + c1 * (np.sin(th) * C[:, 0] - np.cos(th) * C[:, 1])


CASES = [(1, 1), (63, 2), (64, 3), (257, 8), (1000, 9), (4097, 16), (70001, 6), (150001, 0), (150001, 5),
         (150001, 16), (300007, 12), (600011, 4)]


@pytest.mark.parametrize("N,K", CASES)
@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_rhs_and_first_steps(km, N, K, prec):
    """f within one rounding of each of its few operations (FP32: 4 ulp of
    1 + |omega| + |coupling|), and three fixed Euler-small DP45 steps
    h = 2^-10 whose phases follow theta + t f to O(t^2 |f'||f|), the scale
    set by the couplings (at most c1 |C|, order 1 here)."""
    dtype, p = (np.float32, km.F32) if prec == "f32" else (np.float64, km.F64)
    theta, om, X, w = _problem(km, N, K, dtype, 7 * N + K)
    print(f"case lowrank N={N} K={K} {prec}", flush=True)
    h = 2.0 ** -10
    with km.Integrator(N, p, atol=1e-6, c1=3.0, fixed=True) as it:
        it.set_omega(om)
        it.set_factor(X, w)
        it.use_factored("contract")
        f = it.rhs(theta)
        it.set_state(theta, 0.0, h)
        it.begin([h, 3 * h], 1.0, keep_rows=True, ring_rows=4)
        it.advance(1)
        f2 = it.rhs(theta)  # between attempts: its own partial buffers
        st = it.advance(2)
        rows, r = it.read_outputs()
        y, t, _ = it.get_state()
    ref = _field(theta, om, X, w, 3.0)
    scale = 1.0 + np.abs(om) + np.abs(ref - om)
    eps = 2.0 ** -24 if prec == "f32" else 2.0 ** -53
    assert np.max(np.abs(f - ref) / scale) < (8 * eps if prec == "f32" else 1e-12)
    assert np.array_equal(f, f2)
    assert st.accepted == 3 and t == 3 * h and len(rows) == 2
    # one DP45 step sequence in double, the same fixed h
    y64 = theta.astype(np.float64)
    for _ in range(3):
        k1 = _field(y64, om, X, w, 3.0)
        k2 = _field(y64 + h / 2 * k1, om, X, w, 3.0)
        k3 = _field(y64 + h / 2 * k2, om, X, w, 3.0)
        k4 = _field(y64 + h * k3, om, X, w, 3.0)
        y64 = y64 + h / 6 * (k1 + 2 * k2 + 2 * k3 + k4)  # order 4: h^5 = 2^-50
    tol = 16 * eps * (3 + 3 * h * np.max(scale)) + 1e-12
    assert np.max(np.abs(y - y64)) < tol
    assert np.max(np.abs(rows[1] - y64)) < tol
    assert abs(r[1] - np.abs(np.mean(np.exp(1j * y64)))) < max(1e-12, 8 * eps)
