"""The packed-sign passes (sign_mfma_kernel) where their cut of the work can go
wrong: the (256-row group, 1024-wide pair) units are cut into equal stretches
over the workgroups, whatever row group a stretch begins or ends in.  Sizes:
with the ones row, exactly one row group and one row more; a single pair and
one k more; stretches of 2 or 3 units that straddle row groups of 3 pairs; more
units than two per resident workgroup (stretches of uneven length).  Against
the oracle's factored path (kuramoto.cu:62-101 restated).  The integer sums are
exact, so each coupling differs from the oracle's by its input rounding
(2^-54) and the oracle's own double rounding: below one unit of the working
precision of the row scale |w_i| + c K, the bounds below (2^-22, 1e-13)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,K,prec", [(255, 1024, "f32"), (256, 1025, "f32"), (1023, 255, "f64"), (2303, 11265, "f32"),
                                      (2304, 3073, "f64"), (1, 1, "f64"), (20000, 16384, "f32")])
def test_sign_passes_cut(km, orc, N, K, prec):
    dtype = np.float32 if prec == "f32" else np.float64
    seed, c1 = 3, 1.5
    rng = np.random.default_rng(N + K)
    omega = rng.standard_normal(N).astype(dtype)
    theta = rng.uniform(-30, 30, N).astype(dtype)
    print(f"case sign passes N={N} K={K} {prec}", flush=True)
    with km.Integrator(N, km.F32 if prec == "f32" else km.F64, c1=c1) as it:
        it.set_omega(omega)
        it.set_factor_sign(K, seed)
        it.use_factored(True)
        f, cp = it.rhs(theta, couplings=True)
        f2, cp2 = it.rhs(theta, couplings=True)
    assert np.array_equal(f, f2) and np.array_equal(cp, cp2)
    X = orc.rademacher_factor(N, K, seed).astype(dtype)
    w = orc.factor_weights(N, K, False, dtype)
    fo, cso = orc.rhs(orc.Adj(2, X=X, w=w), omega, c1, theta, dtype=dtype)
    tol = (2.0**-22 if prec == "f32" else 1e-13) * (np.abs(omega.astype(np.float64)) + c1 * K)
    assert np.all(np.abs(f.astype(np.float64) - fo) <= tol)
    assert np.all(np.abs(cp.astype(np.float64) - cso) <= np.repeat(tol, 2))


@pytest.mark.parametrize("N,K", [(255, 257), (513, 1100)])
def test_sign_attempts_with_right_hand_sides_between(km, N, K):
    """The digits of an attempt's vectors are written by the launches that form
    them and stay valid while stand-alone right-hand sides of other phases run
    in between: the same bits as without them."""
    rng = np.random.default_rng(N)
    omega = rng.standard_normal(N).astype(np.float32)
    theta = rng.uniform(-3, 3, N).astype(np.float32)
    out = []
    for between in (False, True):
        print(f"case sign attempts N={N} K={K} between={between}", flush=True)
        with km.Integrator(N, km.F32, atol=1e-7, c1=2.0) as it:
            it.set_omega(omega)
            it.set_factor_sign(K, 5)
            it.use_factored(True)
            it.set_state(theta, 0.0, 1e-3)
            it.begin(np.zeros(0), 10.0)
            for _ in range(4):
                if between:
                    it.rhs(theta[::-1].copy())
                status = it.advance(5)
            out.append((it.get_state()[0], status.accepted, it.rhs(theta)))
    assert np.array_equal(out[0][0], out[1][0]) and out[0][1] == out[1][1]
    assert np.array_equal(out[0][2], out[1][2])
