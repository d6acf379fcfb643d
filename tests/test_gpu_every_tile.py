"""Every kernel of the wide tiles, of plans and of batches, and of the swept rows
against the oracle, bit for bit (tile_cases.py; test_tile_cases.py shows which
kernels they launch)."""
import os

import numpy as np
import pytest

import tile_cases as tc

pytestmark = pytest.mark.gpu

THREADS = max(1, min(16, len(os.sched_getaffinity(0)) if hasattr(os, "sched_getaffinity") else 1))


def _case(orc, eq, bc, n, prec, steps, dt, dx=None):
    """The initial state and the oracle's after `steps`."""
    dtype = np.float64 if prec == 0 else np.float32
    rng = np.random.default_rng(n + steps)
    if eq == 0:
        u0 = (1.0 + 0.1 * rng.standard_normal(n)).astype(dtype)  # the ends differ from their neighbours
        fo, fo2 = orc.heat_consts(dt, dtype) if dx is None else orc.heat_consts(dt, dtype, ds=dx)
        return u0, orc.heat_run(u0, steps, fo, fo2, 1 if bc == 2 else 0, THREADS)
    if eq == 1:
        u0 = orc.ic_ks_noisy(n, 3).astype(dtype)
        return u0, orc.ks_run(u0, steps, orc.ks_consts(dt, dtype), THREADS)
    u0 = orc.euler_ic_ref(n, dtype)
    u0.reshape(n, 3)[1:-1] *= (1 + 0.01 * rng.random((n - 2, 1))).astype(dtype)
    k, bd = orc.euler_consts(dt, n, dtype)
    return u0, orc.euler_run(u0, steps, k, bd, THREADS)


def _dt(eq, n):
    return 0.1 / (n - 2) if eq == 2 else (0.005 if eq == 1 else 0.001)


def _same(got, want):
    bad = np.flatnonzero(got != want)
    assert bad.size == 0, f"{bad.size} mismatches, first at {bad[:8]}"


@pytest.mark.parametrize("eq,prec,n,steps,bc", [c + (0,) for c in tc.PLANS] + [c + (2,) for c in tc.PLANS if c[0] == 0])
def test_plan_tiles(sw, orc, eq, prec, n, steps, bc):
    print(f"plan tile eq={eq} prec={prec} n={n} steps={steps} bc={bc}", flush=True)
    u0, want = _case(orc, eq, bc, n, prec, steps, _dt(eq, n))
    with sw.Plan(eq, n, _dt(eq, n), precision=prec, algorithm=sw.TRAPEZOID, node_width=128, bc=bc) as p:
        p.set_state(u0)
        p.advance(steps)
        _same(p.get_state(), want)


@pytest.mark.parametrize("eq,prec,n,steps", tc.BATCHES)
def test_batch_tiles(sw, orc, eq, prec, n, steps):
    dt, dx = (0.001, 0.001) if eq == 0 else (0.005, 0.5)
    print(f"batch tile eq={eq} prec={prec} n={n} steps={steps}", flush=True)
    u0, want = _case(orc, eq, 2, n, prec, steps, dt, dx if eq == 0 else None)
    one = np.full(1, eq, np.int32), np.full(1, n, np.int64), np.full(1, dt), np.full(1, dx)
    with sw.Batch(*one, precision=prec) as b:
        b.set_state(u0)
        b.advance(steps)
        _same(b.get_state(), want)


@pytest.mark.parametrize("eq,bc,prec,W,n", tc.ROWS)
def test_swept_rows(sw, orc, eq, bc, prec, W, n):
    steps = tc.row_steps(eq, W)
    print(f"swept rows eq={eq} bc={bc} prec={prec} W={W} n={n} steps={steps}", flush=True)
    u0, want = _case(orc, eq, bc, n, prec, steps, _dt(eq, n))
    with sw.Plan(eq, n, _dt(eq, n), precision=prec, algorithm=sw.SWEPT, bc=bc, tpb=W, node_width=W) as p:
        p.set_profiling(True)
        p.set_state(u0)
        p.advance(steps)
        assert [p.kernel_stats(k)[0] for k in (sw.K_UP, sw.K_SPLIT, sw.K_DIAMOND, sw.K_DOWN)] == [1, 1, 1, 1]
        _same(p.get_state(), want)


@pytest.mark.parametrize("eq,prec,alg,W,n", tc.PLAIN_ROWS)
def test_swept_rows_without_profiling(sw, orc, eq, prec, alg, W, n):
    steps = tc.row_steps(eq, W)
    print(f"plain rows eq={eq} prec={prec} alg={alg} W={W} n={n} steps={steps}", flush=True)
    u0, want = _case(orc, eq, 0, n, prec, steps, _dt(eq, n))
    with sw.Plan(eq, n, _dt(eq, n), precision=prec, algorithm=alg, tpb=W, node_width=W) as p:
        p.set_state(u0)
        p.advance(steps)
        _same(p.get_state(), want)
