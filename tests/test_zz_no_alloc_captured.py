"""sw1d_advance_noalloc captured into a graph (after its first call on the device):
every replay advances the caller's state by the captured steps once more, also when
another problem has used the workspace in between."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("eq,prec,alg,n,steps", [(0, 0, 0, 4096, 35), (1, 0, 0, 4096, 70), (2, 1, 0, 2048, 5),
                                                 (0, 1, 1, 4096, 129), (1, 0, 1, 8192, 1), (1, 1, 3, 5001, 77),
                                                 (2, 0, 3, 1 << 14, 21)])
def test_replays_continue(sw, orc, eq, prec, alg, n, steps):
    hip = C.CDLL("libamdhip64.so")
    L = sw.lib()
    L.sw1d_advance_noalloc.argtypes = [C.c_void_p, C.c_void_p, C.c_int64, C.c_void_p]
    dtype = np.float64 if prec == 0 else np.float32
    print(f"captured noalloc eq={eq} alg={alg} n={n} steps={steps}", flush=True)
    if eq == 0:
        dt, u0 = 1e-3, orc.heat_ic_ref(n, dtype)
        after = lambda k: orc.heat_run(u0, k, *orc.heat_consts(dt, dtype), 0, 8)
    elif eq == 1:
        dt, u0 = 0.005, orc.ic_ks_noisy(n, 3).astype(dtype)
        after = lambda k: orc.ks_run(u0, k, orc.ks_consts(dt, dtype), 8)
    else:
        dt = 0.1 / (n - 2)
        u0 = orc.euler_ic_ref(n, dtype)
        c, bd = orc.euler_consts(dt, n, dtype)
        after = lambda k: orc.euler_run(u0, k, c, bd, 8)
    prob = sw.Problem(eq, prec, alg, 0, n, 128, 128 if alg else 0, dt, 0.0, 0.0, 0, 0)
    other = sw.Problem(sw.KS, sw.F64, sw.SWEPT, 0, 4096, 128, 128, 0.005, 0.0, 0.0, 0, 0)
    v = orc.ic_ks_noisy(4096, 9)

    def device(a):
        d = C.c_void_p()
        assert hip.hipMalloc(C.byref(d), C.c_size_t(a.nbytes)) == 0
        assert hip.hipMemcpy(d, C.c_void_p(a.ctypes.data), C.c_size_t(a.nbytes), 1) == 0
        return d

    def host(d, like):
        out = np.empty_like(like)
        assert hip.hipMemcpy(C.c_void_p(out.ctypes.data), d, C.c_size_t(out.nbytes), 2) == 0
        return out

    d, e = device(u0), device(v)
    stream, graph, exe = C.c_void_p(), C.c_void_p(), C.c_void_p()
    assert hip.hipStreamCreateWithFlags(C.byref(stream), 1) == 0
    assert L.sw1d_advance_noalloc(C.byref(other), e, 3, stream) == 0
    assert hip.hipStreamBeginCapture(stream, 1) == 0
    assert L.sw1d_advance_noalloc(C.byref(prob), d, steps, stream) == 0
    assert hip.hipStreamEndCapture(stream, C.byref(graph)) == 0
    assert hip.hipGraphInstantiate(C.byref(exe), graph, None, None, C.c_size_t(0)) == 0
    assert np.array_equal(host(d, u0), u0)
    for k in range(1, 4):
        assert hip.hipGraphLaunch(exe, stream) == 0
        assert L.sw1d_advance_noalloc(C.byref(other), e, 5, stream) == 0
        assert hip.hipStreamSynchronize(stream) == 0
        assert np.array_equal(host(d, u0), after(k * steps)), k
    assert np.array_equal(host(e, v), orc.ks_run(v, 18, orc.ks_consts(0.005), 8))
    assert hip.hipGraphExecDestroy(exe) == 0 and hip.hipGraphDestroy(graph) == 0
    assert hip.hipStreamDestroy(stream) == 0
    hip.hipFree(d)
    hip.hipFree(e)
