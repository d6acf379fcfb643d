"""Training sets from batches whose state takes as long to copy as an advance takes:
every pair and the scales against snapshots taken one by one."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,B,nsnap,k", [(1024, 4096, 1, 2), (1024, 4096, 3, 1), (256, 8192, 2, 2), (128, 3, 4, 7)])
def test_pairs_are_the_snapshots(sw, nx, B, nsnap, k):
    rng = np.random.default_rng(nx + B)
    args = (np.ones(B, np.int32), np.full(B, nx, np.int64), np.full(B, 0.005), np.full(B, 0.5))
    u0 = rng.standard_normal(B * nx)
    print(f"dataset nx={nx} B={B} nsnap={nsnap}", flush=True)
    with sw.Batch(*args) as b:
        b.set_state(u0)
        snaps = [u0.reshape(B, nx)]
        for _ in range(nsnap):
            b.advance(k)
            snaps.append(b.get_state().reshape(B, nx))
        b.set_state(u0)
        with sw.Surrogate(nx, 2, seed=0) as nn:
            samples, scales = nn.dataset(b, nsnap, k)
            x, t = nn.dataset_samples(0, samples)
    assert samples == nsnap * B
    # sums of B nx nsnap squares in FP64, in another order
    for got, want in zip(scales, (np.array(snaps[:-1]), np.diff(np.array(snaps), axis=0))):
        assert abs(got / np.sqrt(np.mean(want ** 2)) - 1) < 1e-12
    for s in range(nsnap):
        assert np.array_equal(x[s * B:(s + 1) * B], (snaps[s] * (1.0 / scales[0])).astype(np.float32))
        assert np.array_equal(t[s * B:(s + 1) * B], ((snaps[s + 1] - snaps[s]) * (1.0 / scales[1])).astype(np.float32))
