"""Rows drained into device memory."""
import ctypes

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


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
