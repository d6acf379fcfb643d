"""Euler stages of waves whose operands need the operators' scaled divisions and
roots, and of waves next to them that do not, against the oracle bit for bit:
densities, momenta and energies far outside the ordinary range, momenta and
pressure differences down to the smallest denormal numbers, zeros of both signs,
and fields that become NaN (a NaN's own bits are not compared)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

N = 4096


def _state(orc, kind, dtype):
    rng = np.random.default_rng(7)
    u = np.empty((N, 3))
    x = np.arange(N) / N
    u[:, 0] = 1.0 - 0.5 * x + 0.05 * np.sin(40 * x)
    u[:, 1] = 0.2 * np.sin(9 * x)
    u[:, 2] = 2.5 - x
    half = slice(1500, 3000)
    tiny = np.finfo(dtype).tiny
    if kind == "small" or kind == "large":  # the whole equation scales
        u[half] *= {("small", np.float64): 1e-40, ("large", np.float64): 1e40, ("small", np.float32): 1e-5,
                    ("large", np.float32): 1e5}[kind, dtype]
    elif kind == "range":  # neighbours of every size
        span = 60 if dtype == np.float64 else 4
        u[half] *= 10.0 ** rng.uniform(-span, span, (1500, 1))
    elif kind == "momenta":  # equal densities and energies: pressure differences of momenta alone
        u[half, 0], u[half, 2] = 1.0, 2.5
        u[half, 1] = 10.0 ** rng.uniform(np.log10(tiny) - 8, -1, 1500) * rng.choice([-1, 1], 1500)
    elif kind == "zeros":
        u[half, 0], u[half, 2] = 1.0, 2.5
        u[half, 1] = np.where(rng.random(1500) < 0.5, 0.0, -0.0)
        u[2000:2100, 1] = tiny / 4
    else:
        u[2000, 0], u[2600, 2] = -1.0, np.inf
    return u.astype(dtype).ravel()


@pytest.mark.parametrize("prec", [0, 1])
@pytest.mark.parametrize("alg", [0, 1, 3])
@pytest.mark.parametrize("kind", ["small", "large", "range", "momenta", "zeros", "nan"])
def test_irregular_euler_states_match_oracle(sw, orc, kind, alg, prec):
    dtype = np.float64 if prec == 0 else np.float32
    steps = 40
    print(f"irregular euler {kind} alg={alg} prec={prec}", flush=True)
    dt = 0.1 / (N - 2)
    u0 = _state(orc, kind, dtype)
    k, bd = orc.euler_consts(dt, N, dtype)
    want = orc.euler_run(u0, steps, k, bd)
    with sw.Plan(2, N, dt, precision=prec, algorithm=alg, tpb=128, node_width=0 if alg == 0 else 128) as p:
        for profiling in (False, True):
            p.set_profiling(profiling)
            p.set_state(u0)
            p.advance(steps)
            got = p.get_state()
            bad = np.flatnonzero(~((got == want) | (np.isnan(got) & np.isnan(want))))
            assert bad.size == 0, f"profiling={profiling}: {bad.size} mismatches, first at {bad[:8]}"
