"""Between kmt_batch_set_instance and the next begin a batch has no run, but
its records: what is left in the rings drains as usual, and what was set stays
set whatever is read in between."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GRID = 0.05 * np.arange(1, 41)


def _batch(km, shared):
    rng = np.random.default_rng(4)
    Ns = [300] * 3 if shared else [300, 77, 401]
    bt = km.Batch(Ns, shared=shared, storage="bf16")
    X = rng.standard_normal((max(Ns), 5)).astype(np.float32)
    for b, n in enumerate(Ns):
        if not shared or b == 0:
            bt.set_factor(-1 if shared else b, X[:n], np.full(5, -1.0 / (5 * n), np.float32))
        bt.set_instance(b, *_vectors(b, n), 1.0 + b)
    return bt


def _vectors(b, n, again=0):
    rng = np.random.default_rng(10 * again + b)
    return rng.standard_normal(n).astype(np.float32), rng.uniform(-3, 3, n).astype(np.float32)


def _read(bt, b, most):
    r, n = np.zeros(most, np.float32), ctypes.c_int()
    assert bt.lib.kmt_batch_read_order(bt.ptr, b, most, r.ctypes.data, ctypes.byref(n)) == 0
    return r[:n.value]


@pytest.mark.parametrize("shared", [True, False])
def test_orders_drain_after_set_instance(km, shared):
    with _batch(km, shared) as bt:
        bt.begin(GRID, 2.0, ring_rows=64)
        while bt.advance(8).active:
            pass
        want = [bt.read_order(b) for b in range(3)]
    assert all(len(w) == 40 for w in want)
    with _batch(km, shared) as bt:
        bt.begin(GRID, 2.0, ring_rows=64)
        while bt.advance(8).active:
            pass
        got = [[_read(bt, b, 2)] for b in range(3)]
        bt.set_instance(1, *_vectors(1, bt.Ns[1], 1), 2.5, 0.25, 0.003)
        for q in range(60):  # bounded: a count that comes back would never end
            for b in range(3):
                got[b].append(_read(bt, b, 2))
        for b in range(3):
            assert np.array_equal(np.concatenate(got[b]), want[b]), b
        _, rec = bt.get_instance(1)
        assert rec["t"] == 0.25 and rec["h"] == np.float32(0.003)
        bt.begin(2.0 + GRID, 2.5, ring_rows=64)
        assert all(len(bt.read_order(b)) == 0 for b in range(3))


@pytest.mark.parametrize("shared", [True, False])
def test_set_instance_survives_reads(km, shared):
    """The run after a restart is the same with and without reads between
    set_instance and begin."""
    def second(read):
        with _batch(km, shared) as bt:
            if read:
                bt.get_instance(0)  # before any run
                _read(bt, 2, 4)
            bt.begin(GRID, 1.0, ring_rows=64)
            while bt.advance(8).active:
                pass
            for b in range(3):
                bt.set_instance(b, *_vectors(b, bt.Ns[b], 2), 3.0 - b, 0.5, 0.002)
                if read:
                    _read(bt, b, 3)
                    bt.get_instance((b + 1) % 3)
            bt.begin(GRID, 1.5, ring_rows=64)
            while bt.advance(8).active:
                pass
            return [bt.read_order(b) for b in range(3)] + [bt.get_instance(b)[0] for b in range(3)]

    for a, b in zip(second(False), second(True)):
        assert np.array_equal(a, b)


def test_factor_changed_during_a_run(km):
    """16-bit storage has a power-of-two scale of its own: a factor set between
    advances keeps its scale through the next advance and begin."""
    def run(change):
        with _batch(km, False) as bt:
            X = np.random.default_rng(9).standard_normal((77, 5)).astype(np.float32)
            w = np.full(5, -16.0 / (5 * 77), np.float32)
            if change == "before":
                bt.set_factor(1, X, w)
            bt.begin(GRID, 2.0, ring_rows=64)
            bt.advance(4)
            if change == "during":
                bt.set_factor(1, X, w)
                bt.advance(1)
            bt.set_instance(1, *_vectors(1, 77, 3), 1.0, 0.0, 0.01)
            bt.begin(GRID, 2.0, ring_rows=64)
            bt.advance(12)
            return bt.get_instance(1)[0]

    assert np.array_equal(run("before"), run("during"))
