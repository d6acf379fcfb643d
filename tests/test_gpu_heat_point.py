"""Classic heat steps around the size where a lane takes 16 bytes instead of one
point (two waves per SIMD in FP64, seven in FP32), with both kinds of end, against
the oracle bit for bit."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bc", [0, 2])
@pytest.mark.parametrize("prec,n", [(p, s + d) for p, s in ((0, 2 << 16), (1, 7 << 16)) for d in (-1, 0, 1)] +
                         [(p, n) for p in (0, 1) for n in (8, 255, 256, 257)])
def test_heat_steps(sw, orc, prec, n, bc):
    dtype = np.float64 if prec == 0 else np.float32
    rng = np.random.default_rng(n)
    u0 = (1.0 + 0.1 * rng.standard_normal(n)).astype(dtype)  # the ends differ from their neighbours
    print(f"heat steps prec={prec} n={n} bc={bc}", flush=True)
    with sw.Plan(sw.HEAT, n, 1e-3, precision=prec, algorithm=sw.CLASSIC, bc=bc) as p:
        p.set_state(u0)
        p.advance(131)
        got = p.get_state()
    fo, fo2 = orc.heat_consts(1e-3, dtype)
    assert np.array_equal(got, orc.heat_run(u0, 131, fo, fo2, 1 if bc == 2 else 0, 8))
