"""Workgroup-wide overlapped tiles (heat and KS plans) against the oracle, bit
for bit: every tile shape of both equations (the sizes pick points per lane 2 ..
21), windows that wrap the field many times, once and not at all, fields that no
tile width divides, insulated ends (reflected windows), and advances of one step,
of a few and of several launches.  The swept rows that per-kernel profiling
times give the same bits as the tiles that run without it."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [256, 1000, 4113, 20011, 50000, 70000, 131072, 200001, 262144, 400003, 524288, 620001, 700001, 800001,
         900001, 1048576, 2097152]
THREADS = max(1, min(16, len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else 1))


def _case(orc, eq, bc, n, dtype, steps):
    """(initial state, plan keywords, state after `steps` by the oracle)"""
    if eq == 1:
        u0 = orc.ic_ks_noisy(n, 3).astype(dtype)
        return u0, {"dt": 0.005}, orc.ks_run(u0, steps, orc.ks_consts(0.005, dtype), THREADS)
    rng = np.random.default_rng(n)
    u0 = (1.0 + 0.1 * rng.standard_normal(n)).astype(dtype)  # the ends differ from their neighbours
    fo, fo2 = orc.heat_consts(0.001, dtype)
    return u0, {"dt": 0.001, "bc": bc}, orc.heat_run(u0, steps, fo, fo2, 0 if bc != 2 else 1, THREADS)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("eq,bc", [(0, 0), (0, 2), (1, 0)])
def test_wide_tiles_match_oracle(sw, orc, eq, bc, prec, n):
    dtype = np.float64 if prec == 0 else np.float32
    pieces = [1, 7, 120]
    print(f"wide tiles eq={eq} bc={bc} prec={prec} n={n}", flush=True)
    u0, kw, want = _case(orc, eq, bc, n, dtype, sum(pieces))
    with sw.Plan(eq, n, precision=prec, algorithm=sw.TRAPEZOID, node_width=128, **kw) as p:
        p.set_state(u0)
        for k in pieces:
            p.advance(k)
        got = p.get_state()
    bad = np.flatnonzero(got != want)
    assert bad.size == 0, f"{bad.size} mismatches, first at {bad[:8]}"


@pytest.mark.parametrize("eq,bc,prec,W,n", [(0, 0, 0, 64, 128), (0, 0, 0, 512, 8192), (0, 2, 1, 256, 4096),
                                            (1, 0, 0, 1024, 8192), (1, 0, 1, 64, 1024), (1, 0, 1, 512, 1 << 20)])
def test_profiled_swept_rows_and_wide_tiles_agree(sw, orc, eq, bc, prec, W, n):
    """A swept plan switching between rows (profiled: up, diamonds, down,
    classic remainder) and wide tiles keeps the oracle's bits."""
    dtype = np.float64 if prec == 0 else np.float32
    H = W // 2 if eq == 0 else W // 8
    pieces = [H + 3, 3 * H + 1, 5]
    print(f"rows and wide tiles eq={eq} bc={bc} prec={prec} W={W} n={n}", flush=True)
    u0, kw, want = _case(orc, eq, bc, n, dtype, 2 * sum(pieces))
    with sw.Plan(eq, n, precision=prec, algorithm=sw.SWEPT, tpb=W, node_width=W, **kw) as p:
        p.set_state(u0)
        for k in pieces:
            p.set_profiling(True)
            p.advance(k)
            assert k < H or p.kernel_stats(sw.K_UP)[0] == 1
            p.set_profiling(False)
            p.advance(k)
        got = p.get_state()
    assert np.array_equal(got, want)
