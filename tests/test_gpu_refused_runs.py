"""Calls that leave no coupling or no run behind: attempts are refused with
KMT_ERR_STATE, never launched on buffers that are not there, and what comes
after works as if they had not been made."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

STATE, MEMORY = -3, -5


def _refused(km, code, call, *args, **kw):
    with pytest.raises(km.KmtError) as e:
        call(*args, **kw)
    assert e.value.code == code, e.value


def _context(km, N, prec):
    p, dtype = (km.F32, np.float32) if prec == "f32" else (km.F64, np.float64)
    rng = np.random.default_rng(N)
    it = km.Integrator(N, p, atol=1e-6, c1=3.0)
    it.set_omega(rng.standard_normal(N).astype(dtype))
    it.set_factor(rng.standard_normal((N, 5)).astype(dtype), np.full(5, -1.0 / (5.0 * N), dtype))
    it.use_factored("contract")
    it.set_state(rng.uniform(-3, 3, N).astype(dtype), 0.0, 0.01)
    return it


@pytest.mark.parametrize("prec", ["f32", "f64"])
@pytest.mark.parametrize("N", [100, 2000])
def test_coupling_taken_away_during_a_run(km, N, prec):
    print(f"case refused N={N} {prec}", flush=True)

    def run(away):
        with _context(km, N, prec) as it:
            it.begin(0.01 * np.arange(1, 500), 1e6, keep_rows=True, ring_rows=500)
            it.advance(7)
            if away:
                it.use_factored(False)  # no dense adjacency was ever built
                _refused(km, STATE, it.advance, 3)
                _refused(km, STATE, it.step)
                _refused(km, STATE, it.time_attempts, 2)
                assert it.advance(0).attempts == 7  # nothing to launch
                it.use_factored("contract")
            it.advance(9)
            return it.read_times() + it.read_outputs() + it.get_state()

    for a, b in zip(run(False), run(True)):
        assert np.array_equal(a, b)


def test_failed_begin_leaves_no_run(km):
    """A ring of 35 TB."""
    print("case failed begin", flush=True)
    N = 2000

    def run(fail):
        with _context(km, N, "f64") as it:
            theta = it.get_state()[0]
            if fail:
                it.begin([0.5], 1e6, ring_rows=4)
                it.advance(3)
                _refused(km, MEMORY, it.begin, [0.5], 1e6, keep_rows=True, ring_rows=2 ** 31 - 1)
                _refused(km, STATE, it.advance, 3)
                _refused(km, STATE, it.read_outputs, 1)
                _refused(km, STATE, it.read_times)
                it.set_state(theta, 0.0, 0.01)
            f = it.rhs(theta)
            it.begin(0.01 * np.arange(1, 500), 1e6, keep_rows=True, ring_rows=500)
            it.advance(9)
            return (f,) + it.read_times() + it.read_outputs() + it.get_state()

    for a, b in zip(run(False), run(True)):
        assert np.array_equal(a, b)


def test_failed_batch_begin_leaves_no_run(km):
    print("case failed batch begin", flush=True)
    B, N = 8, 2000
    rng = np.random.default_rng(1)
    with km.Batch([N] * B, shared=False, storage="bf16") as bt:
        for b in range(B):
            bt.set_factor(b, rng.standard_normal((N, 5)).astype(np.float32), np.full(5, -1.0 / (5.0 * N), np.float32))
            bt.set_instance(b, rng.standard_normal(N).astype(np.float32),
                            rng.uniform(-3, 3, N).astype(np.float32), 2.0)
        bt.begin(0.01 * np.arange(1, 100), 1e6, ring_rows=100)
        bt.advance(4)
        _refused(km, MEMORY, bt.begin, [0.5], 1e6, ring_rows=2 ** 31 - 1)
        _refused(km, STATE, bt.advance, 1)
        bt.ring_rows = 4
        assert len(bt.read_order(0)) == 0
        bt.begin(0.01 * np.arange(1, 100), 1e6, ring_rows=100)
        assert bt.advance(4).accepted > 0
