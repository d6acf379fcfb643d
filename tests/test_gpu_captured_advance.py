"""Advances captured from a plan's stream into a graph: every replay
advances the state by the captured steps once more, whatever number of launches
those take, also with eager calls between the replays."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


class Captured:
    """What a program's own calls on `stream` between begin and end make a graph."""

    def __init__(self, stream, work):
        self.hip = C.CDLL("libamdhip64.so")
        self.stream, graph, self.exec = C.c_void_p(stream), C.c_void_p(), C.c_void_p()
        assert self.hip.hipStreamBeginCapture(self.stream, 1) == 0  # thread-local
        work()
        assert self.hip.hipStreamEndCapture(self.stream, C.byref(graph)) == 0
        assert self.hip.hipGraphInstantiate(C.byref(self.exec), graph, None, None, C.c_size_t(0)) == 0
        assert self.hip.hipGraphDestroy(graph) == 0

    def replay(self):
        assert self.hip.hipGraphLaunch(self.exec, self.stream) == 0

    def close(self):
        assert self.hip.hipGraphExecDestroy(self.exec) == 0


def _case(orc, eq, n, dtype):
    """(initial state, time step, steps -> the oracle's state)"""
    if eq == 1:
        u0 = orc.ic_ks_noisy(n, 3).astype(dtype)
        return u0, 0.005, lambda k: orc.ks_run(u0, k, orc.ks_consts(0.005, dtype), 8)
    if eq == 0:
        u0 = orc.heat_ic_ref(n, dtype)
        fo, fo2 = orc.heat_consts(0.001, dtype)
        return u0, 0.001, lambda k: orc.heat_run(u0, k, fo, fo2, 0, 8)
    dt = 0.1 / (n - 2)
    u0 = orc.euler_ic_ref(n, dtype)
    k, bd = orc.euler_consts(dt, n, dtype)
    return u0, dt, lambda s: orc.euler_run(u0, s, k, bd, 8)


@pytest.mark.parametrize("steps", [1, 2, 35, 70, 129])
@pytest.mark.parametrize("eq,alg,W,n,prec", [(0, 0, 0, 4096, 0), (1, 0, 0, 4099, 1), (2, 0, 0, 2048, 0),
                                             (0, 1, 128, 4096, 1), (1, 1, 128, 4096, 0), (2, 1, 128, 4096, 0),
                                             (1, 2, 128, 4096, 0), (0, 3, 128, 4096, 0), (1, 3, 128, 4099, 0),
                                             (2, 3, 128, 4097, 1), (1, 1, 512, 1 << 20, 1)])
def test_replays_continue(sw, orc, eq, alg, W, n, prec, steps):
    u0, dt, after = _case(orc, eq, n, np.float64 if prec == 0 else np.float32)
    print(f"captured advance eq={eq} alg={alg} n={n} steps={steps}", flush=True)
    with sw.Plan(eq, n, dt, precision=prec, algorithm=alg, tpb=W or 64, node_width=W) as p:
        p.set_state(u0)
        p.advance(70)  # a classic plan has its own graph then
        p.set_state(u0)
        g = Captured(p.stream(), lambda: p.advance(steps))
        p.synchronize()
        assert np.array_equal(p.get_state(), u0)  # nothing ran yet
        for k in range(1, 4):
            g.replay()
            p.synchronize()
            assert np.array_equal(p.get_state(), after(k * steps)), k
        g.replay()
        g.replay()
        assert np.array_equal(p.get_state(), after(5 * steps))
        p.advance(1)
        g.replay()
        p.advance(70)
        g.replay()
        assert np.array_equal(p.get_state(), after(7 * steps + 71))
        p.set_state(u0)
        g.replay()
        assert np.array_equal(p.get_state(), after(steps))
        g.close()

