"""Loss and gradient of the surrogate at the sizes where their tiles have edges:
one 64-position tile, samples that the 256-position tile does not divide, and
position shares that are uneven or empty (the weight gradients split the
positions over up to 64 workgroups and two waves each), against the CPU oracle
with the device's BF16 roundings.  Tolerances: those of the gradient test at
nx = 1024 (BF16 gradients between layers, FP32 sums)."""
import numpy as np
import pytest

import nn_oracle as no

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,batch", [(64, 1), (64, 3), (128, 5), (192, 1), (192, 23), (256, 1), (512, 9), (1280, 3)])
def test_gradient_at_tile_edges(sw, nx, batch):
    rng = np.random.default_rng(1000 * nx + batch)
    x = rng.standard_normal((batch, nx)).astype(np.float32)
    t = (0.3 * rng.standard_normal((batch, nx))).astype(np.float32)
    p = (rng.standard_normal(no.NPARAM) * 0.25 / np.sqrt(8)).astype(np.float32)
    print(f"surrogate gradient nx={nx} batch={batch}", flush=True)
    with sw.Surrogate(nx, batch + 1, seed=0) as nn:
        nn.set_params(p)
        loss, g = nn.gradient(x, t)
        again = nn.gradient(x, t)
    assert again[0] == loss and np.array_equal(again[1], g)  # fixed summation order
    wl, wg = no.loss_grad(p.astype(np.float64), x, t, bf=True)
    assert abs(loss - wl) < 1e-3 * wl
    o = 0
    for name, shape in no.SIZES:
        k = int(np.prod(shape))
        rel = np.linalg.norm(g[o:o + k] - wg[o:o + k]) / np.linalg.norm(wg[o:o + k])
        assert rel < 3e-2, (name, rel)
        o += k
