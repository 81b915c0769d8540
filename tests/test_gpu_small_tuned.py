"""Tuning and timing know the one-workgroup form of small dense networks: a
tuned context's attempts stay in it, and timed attempts are those that
advances run."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _context(km, prec, N):
    dtype, p, atol = (np.float32, km.F32, 1e-6) if prec == "f32" else (np.float64, km.F64, 1e-9)
    rng = np.random.default_rng(N)
    it = km.Integrator(N, p, atol=atol, c1=3.0)
    it.set_omega(np.tan(np.pi * (rng.random(N) - 0.5)).astype(dtype))
    it.set_factor(rng.standard_normal((N, 5)).astype(dtype), np.full(5, -1.0 / (5.0 * N), dtype))
    it.build_adjacency("native")
    it.set_state(rng.uniform(-3, 3, N).astype(dtype), 0.0, 0.01)
    return it


def _run(it, timed):
    it.begin(0.01 * np.arange(1, 3000), 1e6, keep_rows=True, ring_rows=3000)
    for _ in range(6):
        if timed:
            it.time_attempts(32)
        else:
            it.advance(32)
    times, hs = it.read_times()
    rows, r = it.read_outputs()
    return (times, hs, rows, r) + it.get_state()


@pytest.mark.parametrize("prec,N", [("f32", 200), ("f32", 256), ("f64", 100), ("f64", 128)])
def test_tuned_and_timed_runs_are_the_same(km, prec, N):
    print(f"case small tuned {prec} N={N}", flush=True)
    runs = []
    for tuned, timed in ((False, False), (True, False), (False, True), (True, True)):
        with _context(km, prec, N) as it:
            if tuned:
                it.autotune(2)
            runs.append(_run(it, timed))
    for other in runs[1:]:
        for a, b in zip(runs[0], other):
            assert np.array_equal(a, b)


@pytest.mark.parametrize("prec,N", [("f32", 200), ("f64", 100)])
def test_tuning_keeps_the_fast_form(km, prec, N):
    """One launch for all attempts against eight each: about half the time."""
    print(f"case small tuned time {prec} N={N}", flush=True)
    ms = {}
    for how in ("tuned", "pinned"):
        with _context(km, prec, N) as it:
            it.autotune(2) if how == "tuned" else it.select_variant(8, nontemporal=False, ring=True)
            it.begin([], 1e6, keep_rows=False, ring_rows=1)
            ms[how] = 1e9
            for _ in range(8):
                region, stage, _ = it.time_attempts(64)
                it.read_times()
                assert 0 < stage <= region / 64
                ms[how] = min(ms[how], region)
    print(ms, flush=True)
    assert ms["tuned"] < 0.8 * ms["pinned"]
