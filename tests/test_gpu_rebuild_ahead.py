"""The K = 5 register-rebuild kernel, whose FP32 form loads one chunk of columns
ahead: sizes around its 1024-column chunks (one thread's first chunk past the
end, exactly one chunk, one column more, two).  The rebuilt entries, their
order and the sums are the dense path's on the generated matrix, so the
right-hand sides and couplings are equal bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N", [1, 17, 960, 1024, 1025, 2048, 2049])
@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_rebuild_k5_equals_dense(km, N, prec):
    dt = np.float32 if prec == "f32" else np.float64
    rng = np.random.default_rng(N)
    omega, theta = rng.standard_normal(N).astype(dt), rng.uniform(-3, 3, N).astype(dt)
    X, w = rng.standard_normal((N, 5)).astype(dt), (rng.standard_normal(5) / N).astype(dt)
    out = []
    for mode in ("rebuild", "dense"):
        print(f"case rebuild K=5 N={N} {prec} {mode}", flush=True)
        with km.Integrator(N, km.F32 if prec == "f32" else km.F64, c1=3.0) as it:
            it.set_omega(omega)
            it.set_factor(X, w)
            if mode == "rebuild":
                it.use_factored("rebuild")
            else:
                it.build_adjacency()
            out.append(it.rhs(theta, couplings=True))
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
