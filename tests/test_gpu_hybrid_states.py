"""The hybrid algorithm, whose boundary node the host computes, on states that differ
in every cell, against the oracle bit for bit (a piecewise constant state leaves most
interfaces without a dissipation whose rounding could show)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eq,W", [(0, 64), (0, 1024), (2, 64), (2, 128), (2, 256), (2, 512)])
@pytest.mark.parametrize("prec", [0, 1])
def test_hybrid_on_uneven_states(sw, orc, eq, W, prec):
    n, H = 8 * W, W // 2 if eq == 0 else W // 8
    dtype = np.float64 if prec == 0 else np.float32
    rng = np.random.default_rng(W)
    print(f"hybrid eq={eq} W={W} prec={prec}", flush=True)
    for steps in (2 * H, 5 * H + 3):
        if eq == 0:
            dt = 1e-3
            u0 = (1.0 + 0.1 * rng.standard_normal(n)).astype(dtype)
            want = orc.heat_run(u0, steps, *orc.heat_consts(dt, dtype), 0, 8)
        else:
            dt = 0.1 / (n - 2)
            u0 = orc.euler_ic_ref(n, dtype)
            u0.reshape(n, 3)[1:-1] *= (1 + 0.01 * rng.random((n - 2, 1))).astype(dtype)
            k, bd = orc.euler_consts(dt, n, dtype)
            want = orc.euler_run(u0, steps, k, bd, 8)
        with sw.Plan(eq, n, dt, precision=prec, algorithm=sw.ALT, tpb=W, node_width=W) as p:
            p.set_state(u0)
            p.advance(steps)
            got = p.get_state()
        bad = np.flatnonzero(got != want)
        assert bad.size == 0, f"steps {steps}: {bad.size} mismatches, first at {bad[:8]}"
