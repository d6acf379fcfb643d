"""A classic step, one launch for both stages, against the oracle bit for bit:
the smallest fields (a wave's window wraps them many times), the edges of a
wave's and a workgroup's points at each number of points per lane, odd sizes
(components that start at no multiple of 16 bytes), and both ends of every
equation.  The launch per stage that profiling times gives the same bits."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# at 1024 SIMDs: KS and Euler 56 points per wave, four waves per workgroup, up to
# 57344 points (Euler 458752), then 120 (FP32 240) points per wave; heat a point
# per thread up to 131072, then 124 (FP32 248) points per wave
KS = [8, 9, 55, 57, 63, 224, 225, 1000, 57343, 57407, 57600, 60001, 65536]
HEAT = [8, 9, 255, 257, 1000, 131071, 131072, 131073, 131130, 131201, 132001]
EULER = [8, 9, 55, 57, 63, 224, 225, 1000, 2049, 458751, 458809, 460801]
CASES = ([(0, bc, n) for bc in (0, 2) for n in HEAT] + [(1, 0, n) for n in KS] + [(2, 0, n) for n in EULER])
THREADS = max(1, min(16, len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else 1))


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("eq,bc,n", CASES)
def test_classic_step_matches_oracle(sw, orc, eq, bc, n, prec):
    dtype = np.float64 if prec == 0 else np.float32
    rng = np.random.default_rng(n)
    steps = [1, 66, 2] if n < 100000 or eq == 0 else [1, 3, 1]
    print(f"classic step eq={eq} bc={bc} prec={prec} n={n}", flush=True)
    if eq == 2:
        kw = {"dt": 0.1 / (n - 2)}
        u0 = orc.euler_ic_ref(n, dtype)
        u0.reshape(n, 3)[1:-1] *= (1 + 0.01 * rng.random((n - 2, 1))).astype(dtype)
        k, bd = orc.euler_consts(kw["dt"], n, dtype)
        want = orc.euler_run(u0, sum(steps), k, bd, THREADS)
    elif eq == 1:
        u0 = orc.ic_ks_noisy(n, 3).astype(dtype)
        want = orc.ks_run(u0, sum(steps), orc.ks_consts(0.005, dtype), THREADS)
        kw = {"dt": 0.005}
    else:
        u0 = (1.0 + 0.1 * rng.standard_normal(n)).astype(dtype)
        fo, fo2 = orc.heat_consts(0.001, dtype)
        want = orc.heat_run(u0, sum(steps), fo, fo2, 0 if bc != 2 else 1, THREADS)
        kw = {"dt": 0.001, "bc": bc}
    with sw.Plan(eq, n, precision=prec, algorithm=sw.CLASSIC, **kw) as p:
        p.set_state(u0)
        p.advance(steps[0])
        p.advance(steps[1])
        p.set_profiling(True)
        p.advance(steps[2])
        assert p.kernel_stats(sw.K_CLASSIC)[0] == steps[2] * (1 if eq == 0 else 2)
        p.set_profiling(False)
        got = p.get_state()
    bad = np.flatnonzero(got != want)
    assert bad.size == 0, f"{bad.size} mismatches, first at {bad[:8]}"
