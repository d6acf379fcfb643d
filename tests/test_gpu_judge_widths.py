"""The judge where a problem's size is no multiple of the 256 points that a
block of the distance's sums takes: each problem is judged on its own points,
and the state it keeps, the fallback count and the largest error agree with the
distances computed on the host."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,B", [(128, 2), (128, 7), (192, 4), (320, 6), (448, 5), (512, 4)])
def test_problems_are_judged_on_their_own_points(sw, nx, B):
    K = 20
    rng = np.random.default_rng(nx + B)
    p = (rng.standard_normal(sw.Surrogate.param_count()) * 0.05).astype(np.float32)
    x = np.arange(nx) * 0.5
    # neighbours of very different amplitude, so of different relative error
    u0 = np.concatenate([(0.2 + 1.5 * (i % 3)) * (np.cos(2 * np.pi * (i + 1) * x / (nx * 0.5)) + 0.3)
                         + 0.01 * rng.standard_normal(nx) for i in range(B)])
    args = (np.ones(B, np.int32), np.full(B, nx, np.int64), np.full(B, 0.005), np.full(B, 0.5))
    print(f"judge nx={nx} B={B}", flush=True)
    with sw.Surrogate(nx, B, seed=0) as nn, sw.Batch(*args) as b, sw.Batch(*args) as ref:
        nn.set_params(p)
        nn.set_scales(1.0, 0.02)
        b.set_state(u0)
        nn.advance(b, 1, K, judge_every=0)
        net = b.get_state().reshape(B, nx)
        ref.set_state(u0)
        ref.advance(K)
        plain = ref.get_state().reshape(B, nx)
        e = np.linalg.norm(net - plain, axis=1) / np.linalg.norm(plain, axis=1)
        order = np.sort(e)
        j = int(np.argmax(np.diff(order)))
        tol = 0.5 * (order[j] + order[j + 1])  # far from every distance
        b.set_state(u0)
        st = nn.advance(b, 1, K, judge_every=1, tol=tol)
        got = b.get_state().reshape(B, nx)
    kept = e <= tol
    assert 0 < kept.sum() < B
    assert st["judged"] == 1 and st["fallbacks"] == int((~kept).sum())
    assert abs(st["max_judged_error"] / e.max() - 1) < 1e-9
    for i in range(B):
        assert np.array_equal(got[i], net[i] if kept[i] else plain[i]), (i, e[i], tol)
