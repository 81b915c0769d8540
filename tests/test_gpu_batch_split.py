"""The shared product's default split-K, the order of its FP32 sums: 8 for
adaptive steps, by the documented rule on N and B for a fixed one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _rule(N, B):
    """The cheapest split of a fixed-step batch (hi + lo vectors)."""
    mt, ldn = -(-2 * B // 32), -(-N // 512) * 512
    nkc, nrb = -(-N // 64), ldn // 256
    t_chunk = 0.6e-6 + 0.34e-6 * mt

    def cost(c):
        return -(-nrb * c // 256) * (-(-nkc // c) * t_chunk + 3e-6) + 2.0 * c * 32 * mt * ldn * 4 / 5e12

    return min(range(1, 17), key=cost)


def _run(km, N, B, fixed, split):
    rng = np.random.default_rng(N + B)
    bt = km.Batch([N] * B, atol=1e-6, shared=True, storage="bf16", fixed=fixed)
    bt.set_factor(-1, rng.standard_normal((N, 5)).astype(np.float32), np.full(5, -1.0 / (5.0 * N), np.float32))
    for b in range(B):
        om = np.tan(np.pi * (rng.random(N) - 0.5)).astype(np.float32)
        bt.set_instance(b, om, rng.uniform(-3, 3, N).astype(np.float32), 0.5 + b, 0.0, 0.01)
    if split:
        bt.select_tile(3, split)
    bt.begin(0.1 * np.arange(1, 100), 1e6, ring_rows=64)
    st = bt.advance(16)
    out = [bt.get_instance(b) for b in range(B)]
    bt.close()
    return st.accepted, st.rejected, out


def _same(a, b):
    return a[:2] == b[:2] and all(np.array_equal(x[0], y[0]) and x[1] == y[1] for x, y in zip(a[2], b[2]))


@pytest.mark.parametrize("N,B", [(300, 2), (2000, 33), (2000, 64), (5000, 12), (20000, 64)])
def test_adaptive_runs_keep_one_split(km, N, B):
    print(f"case split N={N} B={B} adaptive, rule {_rule(N, B)}", flush=True)
    assert _same(_run(km, N, B, False, 0), _run(km, N, B, False, 8))


@pytest.mark.parametrize("N,B", [(300, 2), (2000, 33), (5000, 12), (20000, 64)])
def test_fixed_steps_take_the_rule(km, N, B):
    print(f"case split N={N} B={B} fixed, rule {_rule(N, B)}", flush=True)
    assert _same(_run(km, N, B, True, 0), _run(km, N, B, True, _rule(N, B)))
