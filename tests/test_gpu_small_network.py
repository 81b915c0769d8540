"""Networks small enough for one workgroup (whole attempts in one launch)
against the launched stage kernels, which a pinned stage variant keeps: the
same bits, at the edges of a wave, of a group of rows and of the path."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(km, prec, N, pinned, normal, ring, chunk):
    dtype, p, atol = (np.float32, km.F32, 1e-6) if prec == "f32" else (np.float64, km.F64, 1e-9)
    rng = np.random.default_rng(N)
    X = rng.standard_normal((N, 5)).astype(dtype)
    om = (rng.standard_normal(N) if normal else np.tan(np.pi * (rng.random(N) - 0.5))).astype(dtype)
    th = rng.uniform(-3, 3, N).astype(dtype)
    with km.Integrator(N, p, atol=atol, c1=3.0) as it:
        it.set_omega(om)
        # an asymmetric matrix: rows and columns must not be mixed up
        it.set_adjacency((X @ np.roll(X, 1, axis=0).T / -(5.0 * N)).astype(dtype))
        if pinned:
            it.select_variant(8, nontemporal=False, ring=True)
        it.set_state(th, 0.0, 0.5)  # the first step is too large: rejections too
        it.begin(0.03125 * np.arange(1, 33), 1.0, keep_rows=True, ring_rows=ring)
        out = {"rows": [], "r": [], "t": [], "h": []}
        for _ in range(2000):
            st = it.advance(chunk)
            rows, r = it.read_outputs(max_rows=ring if chunk > 1 else 1)
            t, h = it.read_times()
            for k, v in zip(("rows", "r", "t", "h"), (rows, r, t, h)):
                out[k].append(v)
            if not st.active:
                break
        out = {k: np.concatenate(v) for k, v in out.items()}
        out["end"] = it.get_state()[0]
        out["eval"] = it.eval(0.99)
        out["counts"] = np.array([st.accepted, st.rejected, st.attempts, st.rhs_evals, st.active])
        f = it.rhs(th)
        it.set_state(th, 0.0, 0.01)
        it.begin([], 1.0, keep_rows=False, ring_rows=1)
        out["step"] = np.array([it.step()[1:] for _ in range(3)])
        out["f"] = f
    return out


@pytest.mark.parametrize("N", [1, 2, 7, 8, 9, 63, 64, 65, 127, 128, 129, 192, 193, 255, 256, 257])
@pytest.mark.parametrize("prec", ["f32", "f64"])
def test_equals_launched_kernels(km, prec, N):
    for normal, ring, chunk in ((True, 64, 32), (False, 2, 16), (True, 1, 1)):
        print(f"case small N={N} {prec} normal={normal} ring={ring} chunk={chunk}", flush=True)
        a = _run(km, prec, N, False, normal, ring, chunk)
        b = _run(km, prec, N, True, normal, ring, chunk)
        assert a["counts"][4] == 0 and len(a["r"]) == 32
        for k in a:
            assert np.array_equal(a[k], b[k]), k
