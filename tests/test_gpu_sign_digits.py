"""The packed-sign couplings digit for digit, where a workgroup's stretch of
(256-row group, 1024-wide pair) units is neither one row group nor as long as
its neighbour's.  The passes add integers, so NumPy's exact sums of the same
fixed-point numbers (2^-54 units) give the same bits: P_m = sum_n X_nm round(2^54
v_n) rounded once to double, G_m = w_m P_m, C_n likewise from G.  A single bit
of one k in one digit is off by at least one unit of 2^-54, FP64 shows every
one; the FP32 outputs are the same doubles rounded."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _phases(km, dtype, n, rng):
    """n phases and the library's own (cos, sin) of them: the couplings of an
    identity matrix."""
    th = rng.uniform(-30, 30, n).astype(dtype)
    with km.Integrator(n, km.F32 if dtype == np.float32 else km.F64) as it:
        it.set_omega(np.zeros(n, dtype))
        it.set_adjacency(np.eye(n, dtype=dtype))
        _, cs = it.rhs(th, couplings=True)
    cs = np.asarray(cs).reshape(n, 2).astype(np.float64)
    ulp = 2.0 ** (-22 if dtype == np.float32 else -51)
    assert np.max(np.abs(cs - np.stack([np.cos(th.astype(float)), np.sin(th.astype(float))], 1))) < ulp
    return th, cs


def _exact_products(blocks, v, out_len, transposed):
    """X^T v (transposed) or X v for integer v below 2^56, exactly, as Python
    integers: 27-bit pieces, whose sums over < 2^20 terms are exact in double."""
    lo = (v & (2 ** 27 - 1)).astype(np.float64)
    hi = (v >> 27).astype(np.float64)
    both = np.concatenate([hi, lo], 1)
    acc = np.zeros((out_len, 4))
    for at, x in blocks():
        x = x.astype(np.float64)
        if transposed:
            acc += x.T @ both[at:at + len(x)]
        else:
            acc[at:at + len(x)] = x @ both
    return [[(int(r[c]) << 27) + int(r[2 + c]) for c in (0, 1)] for r in acc]


@pytest.mark.parametrize("N,K", [(2304, 3073), (20000, 16384), (9000, 40000)])
@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_couplings_digit_for_digit(km, orc, N, K, prec):
    dtype = np.float32 if prec == "f32" else np.float64
    seed, c1 = 11, 1.5
    rng = np.random.default_rng(N + K)
    print(f"case sign digits N={N} K={K} {prec}", flush=True)
    th, cs = _phases(km, dtype, 1500, rng)
    pick = rng.integers(0, 1500, N)
    omega = rng.standard_normal(N).astype(dtype)
    with km.Integrator(N, km.F32 if prec == "f32" else km.F64, c1=c1) as it:
        it.set_omega(omega)
        it.set_factor_sign(K, seed)
        it.use_factored(True)
        f, cpl = it.rhs(th[pick], couplings=True)
    X = orc.rademacher_factor(N, K, seed)
    w = orc.factor_weights(N, K, False, dtype).astype(np.float64)

    def blocks():
        for a in range(0, N, 1000):
            yield a, X[a:a + 1000]

    v = np.rint(cs[pick] * 2.0 ** 54).astype(np.int64)
    P = np.array([[float(q) for q in r] for r in _exact_products(blocks, v, K, True)]) * 2.0 ** -54
    G = np.rint(P * w[:, None] * 2.0 ** 54).astype(np.int64)
    C = np.array([[float(q) for q in r] for r in _exact_products(blocks, G, N, False)]) * 2.0 ** -54
    assert np.array_equal(np.asarray(cpl).reshape(N, 2), C.astype(dtype))
    # f = omega + c1 (sin C - cos S): four roundings, each of at most the sum of the magnitudes
    c, s = cs[pick].T
    want = omega + c1 * (s * C[:, 0] - c * C[:, 1])
    scale = np.abs(omega) + c1 * (np.abs(C[:, 0]) + np.abs(C[:, 1]))
    assert np.all(np.abs(f - want) <= 6 * (2.0 ** -24 if prec == "f32" else 2.0 ** -53) * scale)
