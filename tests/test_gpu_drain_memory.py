"""Where drains go and what they take: rows into device memory, batch rings
that hold more than the pinned stage."""
import ctypes
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _mapped():
    """Bytes of this process's address space."""
    with open("/proc/self/statm") as f:
        return int(f.read().split()[0]) * os.sysconf("SC_PAGE_SIZE")


@pytest.mark.parametrize("N", [63, 5001])
def test_rows_into_device_memory(km, N):
    print(f"case rows to device N={N}", flush=True)

    def context():
        rng = np.random.default_rng(3)
        it = km.Integrator(N, km.F64, fixed=True, c1=3.0)
        it.set_omega(rng.standard_normal(N))
        it.set_factor(rng.standard_normal((N, 1)), np.array([-1.0 / N]))
        it.use_factored("contract")
        it.set_state(rng.uniform(-3, 3, N), 0.0, 0.125)
        it.begin(0.0625 * np.arange(1, 33), 2.0, keep_rows=True, ring_rows=64)
        it.advance(32)
        return it

    with context() as it:
        rows, _ = it.read_outputs()
    hip = ctypes.CDLL("libamdhip64.so.7")
    dev, out = ctypes.c_void_p(), np.zeros((32, N))
    assert hip.hipMalloc(ctypes.byref(dev), ctypes.c_size_t(out.nbytes)) == 0
    with context() as it:
        got = 0
        while got < 32:
            n = ctypes.c_int()
            assert it.lib.kmt_read_outputs(it.ctx, 5, dev.value + got * N * 8, None, ctypes.byref(n)) == 0
            got += n.value
    assert hip.hipMemcpy(ctypes.c_void_p(out.ctypes.data), dev, ctypes.c_size_t(out.nbytes), 2) == 0
    assert hip.hipFree(dev) == 0
    assert np.array_equal(out, rows)


def _batch(km, ring):
    rng = np.random.default_rng(8)
    bt = km.Batch([64, 40], shared=False, storage="bf16", fixed=True)
    for b, n in enumerate(bt.Ns):
        bt.set_factor(b, rng.standard_normal((n, 5)).astype(np.float32), np.full(5, -1.0 / (5 * n), np.float32))
        bt.set_instance(b, rng.standard_normal(n).astype(np.float32), rng.uniform(-3, 3, n).astype(np.float32), 2.0,
                        0.0, 0.125)
    bt.begin(np.arange(1, 150001) * 2.0 ** -18, 0.5, ring_rows=ring)
    return bt


def test_full_rings_and_short_ones(km):
    """131072 values per ring (1 MB in all and more) against rings of 4096."""
    print("case batch rings", flush=True)
    got = [[], []]
    with _batch(km, 4096) as bt:
        for _ in range(200):
            st = bt.advance(1)
            for b in (1, 0):
                got[b].append(bt.read_order(b))
            if not st.active:
                break
    with _batch(km, 150000) as bt:
        while bt.advance(4).active:
            pass
        r, n = np.zeros(150000, np.float32), ctypes.c_int()
        for b in (0, 1):
            assert len(np.concatenate(got[b])) == 131072
            at = 0
            for most in (1, 100000, 150000):
                assert bt.lib.kmt_batch_read_order(bt.ptr, b, most, r[at:].ctypes.data, ctypes.byref(n)) == 0
                at += n.value
            assert at == 131072
            assert np.array_equal(r[:at], np.concatenate(got[b]))


def test_large_rings_take_no_host_memory(km):
    """A ring is a bound, not what a drain holds: reading a few values of rings
    of 2^25 does not pin their 256 MB."""
    print("case large rings", flush=True)
    with _batch(km, 64) as bt:
        bt.advance(1)
        bt.read_order(0)
    with _batch(km, 1 << 25) as bt:
        r, n = np.zeros(16, np.float32), ctypes.c_int()
        bt.advance(1)
        before = _mapped()
        assert bt.lib.kmt_batch_read_order(bt.ptr, 0, 16, r.ctypes.data, ctypes.byref(n)) == 0 and n.value == 16
        print("grew by", _mapped() - before, flush=True)
        assert _mapped() - before < 64 << 20
