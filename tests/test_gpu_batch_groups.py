"""Batches as groups of tiles, against the oracle bit for bit: batches that fill
the chip and that do not, problems below one tile and of many, one equation
only, and step counts below, at and above two launches (launches come in even
numbers, so one step is a launch of one step and one of none)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("count,lo,hi,only", [(1, 16.0, 16.1, 1), (1, 7.0, 7.01, 0), (3, 7.0, 8.0, None),
                                              (700, 7.0, 9.0, None), (40, 12.0, 16.0, None), (30, 14.0, 15.0, 0),
                                              (256, 10.0, 10.0001, 1)])
def test_batch_groups_match_oracle(sw, orc, prec, count, lo, hi, only):
    import importlib

    wl = importlib.import_module("1dsweptcuda_amd.workloads")
    eq, nx, dt, dx = wl.batch_problems(count, seed=17, lo=lo, hi=hi)
    if only is not None:
        eq[:] = only
        dx = np.where(eq == 0, 1.0 / nx, 0.5)
        dt = np.where(eq == 0, 0.4 * dx * dx / wl.ALPHA, 1.6 / (16.0 / dx ** 4 - 4.0 / dx ** 2))
    dtype = np.float64 if prec == 0 else np.float32
    ics = [u.astype(dtype) for u in wl.batch_ics(eq, nx, dx)]
    pieces = [1, 2, 3, 150, 20]
    print(f"batch groups prec={prec} count={count} sizes={nx.min()}..{nx.max()}", flush=True)
    with sw.Batch(eq, nx, dt, dx, precision=prec) as b:
        b.set_state(np.concatenate(ics))
        for k in pieces:
            b.advance(k)
        got = b.split(b.get_state())
    steps = sum(pieces)
    for i in range(count):
        if eq[i] == 0:
            fo, fo2 = orc.heat_consts(dt[i], dtype, ds=dx[i])
            want = orc.heat_run(ics[i], steps, fo, fo2, 1)
        else:
            want = orc.ks_run(ics[i], steps, orc.ks_consts(dt[i], dtype, dx=dx[i]))
        assert np.array_equal(got[i], want), (i, int(eq[i]), int(nx[i]))
