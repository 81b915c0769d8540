"""Draining outputs in pieces, through the pinned staging (several halves),
into pinned memory and between advances gives what one drain gives."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _context(km, N, ring):
    rng = np.random.default_rng(3)
    it = km.Integrator(N, km.F64, fixed=True, c1=3.0)
    it.set_omega(rng.standard_normal(N))
    it.set_factor(rng.standard_normal((N, 1)), np.array([-1.0 / N]))
    it.use_factored("contract")
    it.set_state(rng.uniform(-3, 3, N), 0.0, 0.125)
    it.begin(0.0625 * np.arange(1, 33), 2.0, keep_rows=True, ring_rows=ring)
    return it


@pytest.mark.parametrize("N", [1, 63, 70001])
def test_rows_in_pieces(km, N):
    print(f"case drains N={N}", flush=True)
    with _context(km, N, 64) as it:
        while it.advance(5).active:
            pass
        rows, r = it.read_outputs()
        t, h = it.read_times()
    assert rows.shape == (32, N) and len(t) == 16
    lib = km.load()
    ptr = ctypes.c_void_p()
    assert lib.kmt_host_alloc(8 * 3 * N, ctypes.byref(ptr)) == 0
    pinned = np.ctypeslib.as_array(ctypes.cast(ptr, ctypes.POINTER(ctypes.c_double)), (3, N))
    got_rows, got_r, got_t = [], [], []
    with _context(km, N, 7) as it:  # a ring that fills up
        for q in range(200):
            st = it.advance(3)
            if q % 2:
                n = ctypes.c_int()
                rr = np.zeros(3)
                assert lib.kmt_read_outputs(it.ctx, 3, ptr, rr.ctypes.data, ctypes.byref(n)) == 0
                got_rows.append(pinned[:n.value].copy())
                got_r.append(rr[:n.value])
            else:
                a, b = it.read_outputs(max_rows=2)
                got_rows.append(a)
                got_r.append(b)
            got_t.append(it.read_times(max_n=1)[0])
            if not st.active and sum(map(len, got_r)) == 32 and sum(map(len, got_t)) == 16:
                break
    lib.kmt_host_free(ptr)
    assert np.array_equal(np.concatenate(got_rows), rows)
    assert np.array_equal(np.concatenate(got_r), r)
    assert np.array_equal(np.concatenate(got_t), t)


@pytest.mark.parametrize("shared", [True, False])
def test_batch_orders_in_pieces(km, shared):
    """kmt_batch_read_order two values at a time between advances, instances
    in turn, against whole drains; and an instance restarted in between."""
    def batch():
        rng = np.random.default_rng(4)
        Ns = [300] * 3 if shared else [300, 77, 401]
        bt = km.Batch(Ns, shared=shared, storage="bf16")
        X = rng.standard_normal((max(Ns), 5)).astype(np.float32)
        for b, n in enumerate(Ns):
            if not shared or b == 0:
                bt.set_factor(-1 if shared else b, X[:n], np.full(5, -1.0 / (5 * n), np.float32))
            bt.set_instance(b, rng.standard_normal(n).astype(np.float32),
                            rng.uniform(-3, 3, n).astype(np.float32), 1.0 + b)
        return bt

    grid = 0.05 * np.arange(1, 41)
    with batch() as bt:
        want = bt.run(grid, 2.0, ring_rows=64)["r"]
        end = [bt.get_instance(b)[0] for b in range(3)]
    got = [[], [], []]
    with batch() as bt:
        bt.begin(grid, 2.0, ring_rows=8)
        for q in range(400):
            st = bt.advance(1 + q % 9)
            b = q % 3
            r, n = np.zeros(2, np.float32), ctypes.c_int()
            assert bt.lib.kmt_batch_read_order(bt.ptr, b, 2, r.ctypes.data, ctypes.byref(n)) == 0
            got[b].append(r[:n.value])
            if st.active == 0 and all(sum(map(len, g)) == 40 for g in got):
                break
        for b in range(3):
            assert np.array_equal(np.concatenate(got[b]), want[b])
            assert np.array_equal(bt.get_instance(b)[0], end[b])
