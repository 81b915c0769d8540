"""A run that comes to the dense form between advances uses the fixed choice of
stage variant from its first attempt on: evaluations in between leave no trace
in it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(km, N, prec, first, then, between):
    p, dtype = (km.F32, np.float32) if prec == "f32" else (km.F64, np.float64)
    rng = np.random.default_rng(N)
    om = np.tan(np.pi * (rng.random(N) - 0.5)).astype(dtype)
    X, w = rng.standard_normal((N, 3)).astype(dtype), np.full(3, -1.0 / (3.0 * N), dtype)
    with km.Integrator(N, p, atol=1e-9 if prec == "f64" else 1e-6, c1=3.0) as it:
        it.set_omega(om)
        it.set_factor(X, w)
        if first == "factored":
            it.build_adjacency(then)
            it.use_factored("contract")
        else:
            it.build_adjacency(first)
        it.set_state(np.zeros(N, dtype), 0.0, 1e-3)
        it.begin(0.002 * np.arange(1, 400), 1.0, keep_rows=True, ring_rows=400)
        it.advance(5)
        if first == "factored":
            it.use_factored(False)
        else:
            it.build_adjacency(then)
        if between == "rhs":
            it.rhs(np.ones(N, dtype))
        elif between == "time":
            it.time_stage_kernel(2)
        it.advance(20)
        flags = it.variant_flags()
        if between == "rhs":
            it.rhs(np.ones(N, dtype))
        it.advance(35)
        times, hs = it.read_times()
        rows, r = it.read_outputs()
        y, t, h = it.get_state()
    return flags, times, hs, rows, r, y, t, h


@pytest.mark.parametrize("prec,N,first,then", [("f64", 3000, "factored", "bf16"), ("f64", 5000, "factored", "f16"),
                                               ("f64", 5000, "factored", "native"), ("f32", 5000, "factored", "native"),
                                               ("f64", 9000, "native", "bf16"), ("f64", 3000, "bf16", "native"),
                                               ("f64", 100, "factored", "native")])
def test_evaluations_leave_a_run_alone(km, prec, N, first, then):
    print(f"case switch {prec} N={N} {first} -> {then}", flush=True)
    want = _run(km, N, prec, first, then, None)
    for between in ("rhs", "time"):
        for a, b in zip(want, _run(km, N, prec, first, then, between)):
            assert np.array_equal(a, b), between
