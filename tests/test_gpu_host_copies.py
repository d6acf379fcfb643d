"""Host copies of plan and batch states and of the network's inputs and results:
around the 1 MB that staging memory holds (below, equal, above), at sizes that
are no multiple of a page, from and into memory at odd addresses, and a batch
whose inputs do not fit beside each other."""
import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

MB = 1 << 20
CASES = [(0, 0, n) for n in (8, 513, MB // 8 - 1, MB // 8, MB // 8 + 1, 400001)]
CASES += [(1, 1, n) for n in (9, MB // 4, MB // 4 + 3)] + [(2, 0, n) for n in (8, 43690, 43691, 131073)]


@pytest.mark.parametrize("eq,prec,n", CASES)
def test_plan_state_round_trip(sw, eq, prec, n):
    dtype = np.float64 if prec == 0 else np.float32
    print(f"host copies eq={eq} prec={prec} n={n}", flush=True)
    count = n * (3 if eq == 2 else 1)
    want = np.random.default_rng(n).standard_normal(count).astype(dtype)
    with sw.Plan(eq, n, 0.1 / (n - 2) if eq == 2 else 0.001, precision=prec, algorithm=sw.CLASSIC) as p:
        for off in (0, 8, 4088):  # directly, then through the same staging memory; at odd addresses
            src = np.zeros(count * want.itemsize + 8192, np.uint8)[off:off + want.nbytes].view(dtype)
            dst = np.full(count * want.itemsize + 8192, 7, np.uint8)
            src[:] = want + dtype(off)
            p.set_state(src)
            sw.lib().sw1d_get_state(p._h, C.c_void_p(dst.ctypes.data + off))
            assert np.array_equal(dst[off:off + want.nbytes].view(dtype), want + dtype(off))
            assert (dst[:off] == 7).all() and (dst[off + want.nbytes:] == 7).all()


@pytest.mark.parametrize("nx", [1000, MB // 8, MB // 8 + 8, 900001])
def test_batch_state_round_trip(sw, nx):
    print(f"batch host copies nx={nx}", flush=True)
    want = np.random.default_rng(nx).standard_normal(nx)
    with sw.Batch(np.ones(1, np.int32), np.array([nx], np.int64), np.array([0.005]), np.array([0.5])) as b:
        for k in range(3):
            b.set_state(want + k)
            assert np.array_equal(b.get_state(), want + k)


@pytest.mark.parametrize("B", [1, 16, 120, 200, 300])
def test_gradient_of_a_batch_equals_that_of_its_samples_in_a_larger_network(sw, B):
    """The same batch with staging memory for it and for a batch far larger
    (which copies directly): equal losses and gradients, bit for bit."""
    nx = 1024
    rng = np.random.default_rng(B)
    x, t = (rng.standard_normal((B, nx)).astype(np.float32) for _ in range(2))
    params = (rng.standard_normal(sw.Surrogate.param_count()) * 0.1).astype(np.float32)
    print(f"gradient host copies B={B}", flush=True)
    got = []
    for most in (B, 2 * B + 3):
        with sw.Surrogate(nx, most, seed=0) as nn:
            nn.set_params(params)
            y = nn.forward(x)
            loss, g = nn.gradient(x, t)
            for _ in range(2):  # directly, then through staging memory
                again = nn.gradient(x, t)
                assert again[0] == loss and np.array_equal(again[1], g)
            assert np.array_equal(nn.forward(x), y)
            got.append((y, loss, g))
    assert np.array_equal(got[0][0], got[1][0]) and got[0][1] == got[1][1] and np.array_equal(got[0][2], got[1][2])
    # the loss of the outputs that forward() returned (float32 sums of 256 squares)
    want = np.mean((got[0][0].astype(np.float64) - t) ** 2)
    assert abs(got[0][1] - want) <= 256 * 2.0 ** -24 * want
