"""Advances of a single step, between longer ones: the classic step, whichever
algorithm the plan has (per-kernel profiling counts it as that), with the oracle's
bits."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eq,alg,n", [(e, a, n) for e in (0, 1, 2) for a, n in ((1, 4096), (3, 1001), (3, 1 << 18))] +
                         [(1, 2, 4096)])
def test_single_steps(sw, orc, eq, alg, n):
    dt = 0.1 / (n - 2) if eq == 2 else (0.005 if eq == 1 else 0.001)
    W = 128
    print(f"single steps eq={eq} alg={alg} n={n}", flush=True)
    if eq == 0:
        u0 = 1.0 + 0.1 * np.random.default_rng(n).standard_normal(n)
        want = orc.heat_run(u0, 11, *orc.heat_consts(dt), 0, 8)
    elif eq == 1:
        u0 = orc.ic_ks_noisy(n, 3)
        want = orc.ks_run(u0, 11, orc.ks_consts(dt), 8)
    else:
        u0 = orc.euler_ic_ref(n, np.float64)
        k, bd = orc.euler_consts(dt, n, np.float64)
        want = orc.euler_run(u0, 11, k, bd, 8)
    with sw.Plan(eq, n, dt, algorithm=alg, tpb=W, node_width=W) as p:
        p.set_state(u0)
        for k in (1, 3, 1, 1, 4):
            p.advance(k)
        p.set_profiling(True)
        p.advance(1)
        stages, tiles = p.kernel_stats(sw.K_CLASSIC)[0], p.kernel_stats(sw.K_DIAMOND)[0]
        got = p.get_state()
    assert np.array_equal(got, want)
    assert stages == (1 if eq == 0 else 2) and tiles == 0
