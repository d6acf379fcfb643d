"""Workgroup-wide overlapped tiles of Euler fields against the oracle, bit for
bit: the sizes and step counts that select each tile shape in both precisions,
fields narrower than a tile's window and many tiles wide, sizes that no tile
width divides, the Dirichlet ends at every position within a lane, and the
swept rows that per-kernel profiling times."""
import os

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SIZES = [256, 257, 258, 259, 260, 1000, 4113, 20011, 70001, 131072, 200003, 262144, 400003, 700001, 1048576]
THREADS = max(1, min(16, len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else 1))


def _case(orc, n, dtype, steps):
    rng = np.random.default_rng(n)
    dt = 0.1 / (n - 2)
    u0 = orc.euler_ic_ref(n, dtype)
    u0.reshape(n, 3)[1:-1] *= (1 + 0.01 * rng.random((n - 2, 1))).astype(dtype)
    k, bd = orc.euler_consts(dt, n, dtype)
    return u0, dt, orc.euler_run(u0, steps, k, bd, THREADS)


@pytest.mark.parametrize("n", SIZES)
@pytest.mark.parametrize("prec", [0, 1])
def test_wide_euler_tiles_match_oracle(sw, orc, prec, n):
    dtype = np.float64 if prec == 0 else np.float32
    pieces = [1, 3, 61 if n < 100000 else 26]
    print(f"wide euler prec={prec} n={n}", flush=True)
    u0, dt, want = _case(orc, n, dtype, sum(pieces))
    with sw.Plan(2, n, dt, precision=prec, algorithm=sw.TRAPEZOID, node_width=128) as p:
        p.set_state(u0)
        for k in pieces:
            p.advance(k)
        got = p.get_state()
    bad = np.flatnonzero(got != want)
    assert bad.size == 0, f"{bad.size} mismatches, first at {bad[:8]}"


@pytest.mark.parametrize("prec,W,n", [(0, 64, 128), (0, 512, 8192), (1, 128, 1024), (1, 256, 4096)])
def test_profiled_swept_rows_and_wide_euler_tiles_agree(sw, orc, prec, W, n):
    dtype = np.float64 if prec == 0 else np.float32
    H = W // 8
    pieces = [H + 3, 3 * H + 1, 5]
    print(f"euler rows and wide tiles prec={prec} W={W} n={n}", flush=True)
    u0, dt, want = _case(orc, n, dtype, 2 * sum(pieces))
    with sw.Plan(2, n, dt, precision=prec, algorithm=sw.SWEPT, tpb=W, node_width=W) as p:
        p.set_state(u0)
        for k in pieces:
            p.set_profiling(True)
            p.advance(k)
            assert k < H or p.kernel_stats(sw.K_UP)[0] == 1
            p.set_profiling(False)
            p.advance(k)
        got = p.get_state()
    assert np.array_equal(got, want)
