"""The stage-7 error partials of a dense run have a grouping of their own, by a
rule on N and the storage, whatever rows per workgroup the other stages take:
the error norm, and so h and the whole sequence of steps, follow from it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(km, N, prec, storage, setup, attempts=60):
    p, dtype = (km.F32, np.float32) if prec == "f32" else (km.F64, np.float64)
    rng = np.random.default_rng(N)
    om = np.tan(np.pi * (rng.random(N) - 0.5)).astype(dtype)
    X = rng.standard_normal((N, 5)).astype(dtype)
    with km.Integrator(N, p, atol=1e-9 if prec == "f64" else 1e-6, c1=3.0) as it:
        it.set_omega(om)
        it.set_factor(X, np.full(5, -1.0 / (5.0 * N), dtype))
        if storage == "rebuild":
            it.use_factored("rebuild")
        else:
            it.build_adjacency(storage)
        setup(it)
        it.set_state(np.zeros(N, dtype), 0.0, 1e-3)
        it.begin(0.002 * np.arange(1, 400), 1.0, keep_rows=False, ring_rows=400)
        it.advance(attempts)
        times, hs = it.read_times()
        _, r = it.read_outputs()
        y, t, h = it.get_state()
    return times, hs, r, y, t, h


def _same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


CASES = [("f64", "native", 257, 8), ("f64", "native", 4096, 8), ("f64", "native", 5000, 8), ("f64", "native", 5657, 8),
         ("f64", "bf16", 200, 16), ("f64", "f16", 3000, 16), ("f64", "bf16", 4096, 4), ("f64", "f16", 8000, 4),
         ("f64", "bf16", 8001, 16), ("f64", "f16", 11000, 16), ("f32", "native", 5000, 4), ("f32", "native", 8000, 8),
         ("f32", "bf16", 9000, 16)]


@pytest.mark.parametrize("prec,storage,N,rows", CASES)
def test_groups_by_rule(km, prec, storage, N, rows):
    """A caller's variant groups the partials by its rows: with the rule's rows
    it gives the default run's bits."""
    print(f"case error groups {prec} {storage} N={N} rows={rows}", flush=True)
    assert _same(_run(km, N, prec, storage, lambda it: None),
                 _run(km, N, prec, storage, lambda it: it.select_variant(rows)))


@pytest.mark.parametrize("N", [4096, 5000, 5656])
def test_fp64_rebuild_is_the_dense_run(km, N):
    """Register-rebuilt tiles give the dense run bit for bit, also where the
    whole matrix stays in the last-level cache."""
    print(f"case rebuild N={N}", flush=True)
    assert _same(_run(km, N, "f64", "native", lambda it: None), _run(km, N, "f64", "rebuild", lambda it: None))
