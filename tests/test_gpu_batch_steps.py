"""A batch's tiles serve any number of steps: sequences of advances whose step
counts change from call to call, below and above what a launch of the first one's
tiles takes, long enough that the tiles are made anew on the way, against the
oracle bit for bit."""
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("count,lo,hi", [(1, 7.0, 7.01), (1, 16.0, 16.1), (60, 7.0, 12.0), (900, 7.0, 9.0)])
@pytest.mark.parametrize("pieces", [[1, 400, 3, 50, 51, 1, 1, 7], [300, 1, 2, 301, 299, 1, 300], [20, 21] * 12])
def test_changing_step_counts(sw, orc, pieces, count, lo, hi, prec):
    wl = importlib.import_module("1dsweptcuda_amd.workloads")
    dtype = np.float64 if prec == 0 else np.float32
    eq, nx, dt, dx = wl.batch_problems(count, seed=23, lo=lo, hi=hi)
    ics = [u.astype(dtype) for u in wl.batch_ics(eq, nx, dx)]
    print(f"batch steps prec={prec} count={count} pieces={pieces[:3]}", flush=True)
    with sw.Batch(eq, nx, dt, dx, precision=prec) as b:
        b.set_state(np.concatenate(ics))
        for k in pieces:
            b.advance(k)
        got = b.split(b.get_state())
    steps = sum(pieces)
    for i in range(0, count, max(1, count // 100)):
        if eq[i] == 0:
            fo, fo2 = orc.heat_consts(dt[i], dtype, ds=dx[i])
            want = orc.heat_run(ics[i], steps, fo, fo2, 1)
        else:
            want = orc.ks_run(ics[i], steps, orc.ks_consts(dt[i], dtype, dx=dx[i]))
        assert np.array_equal(got[i], want), (i, int(eq[i]), int(nx[i]))
