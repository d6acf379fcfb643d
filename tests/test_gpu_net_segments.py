"""Whole-network inference by segments of a sample: batches on both sides of
each change of the segments' length (128, 256 and 512 positions, 256 CUs), one
sample, and more samples than fit the GPU at once, other multiples of 256
positions, against the per-layer launches bit for bit; and rollouts whose states alternate between two arrays,
against the same steps taken one call at a time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

NX = 1024


def _params(sw, seed):
    return (np.random.default_rng(seed).standard_normal(sw.Surrogate.param_count()) * 0.1).astype(np.float32)


@pytest.mark.parametrize("NX,B", [(1024, b) for b in (1, 32, 96, 97, 128, 129, 160, 161, 192, 193, 256, 257, 513)] +
                         [(256, 1), (256, 300), (256, 1100), (512, 5), (512, 600), (768, 3), (768, 301), (1280, 70),
                          (2048, 2), (2048, 130), (5120, 60)])
def test_segments_match_per_layer_launches(sw, NX, B):
    rng = np.random.default_rng(B)
    x = rng.standard_normal((B, NX)).astype(np.float32)
    u0 = rng.standard_normal(B * NX)
    print("segments", NX, B, flush=True)
    out = {}
    with sw.Surrogate(NX, B, seed=0) as nn:
        nn.set_params(_params(sw, 5))
        nn.set_scales(1.3, 0.07)
        for mode in (nn.INFER_AUTO, nn.INFER_PER_LAYER):
            nn.set_inference(mode)
            y = nn.forward(x)
            with sw.Batch(np.ones(B, np.int32), np.full(B, NX, np.int64), np.full(B, 0.005), np.full(B, 0.5)) as b:
                b.set_state(u0)
                nn.advance(b, 3, 20, judge_every=0)
                out[mode] = (y, b.get_state())
    whole, layers = out[nn.INFER_AUTO], out[nn.INFER_PER_LAYER]
    assert np.array_equal(whole[0].view(np.uint32), layers[0].view(np.uint32))
    assert np.array_equal(whole[1].view(np.uint64), layers[1].view(np.uint64))


@pytest.mark.parametrize("steps,judge", [(1, 0), (2, 0), (5, 0), (7, 1), (7, 2), (8, 3)])
@pytest.mark.parametrize("tol", [1e30, 0.0])
def test_rollout_equals_its_steps(sw, steps, judge, tol):
    """tol = 1e30 keeps every judged network step, 0 replaces it by the solver's."""
    B, k = 3, 10
    u0 = np.random.default_rng(8).standard_normal(B * NX)
    print("rollout", steps, judge, tol, flush=True)
    with sw.Surrogate(NX, B, seed=0) as nn:
        nn.set_params(_params(sw, 6))
        nn.set_scales(1.1, 0.05)
        kinds = (np.ones(B, np.int32), np.full(B, NX, np.int64), np.full(B, 0.005), np.full(B, 0.5))
        with sw.Batch(*kinds) as one, sw.Batch(*kinds) as ref:
            one.set_state(u0)
            nn.advance(one, steps, k, judge_every=judge, tol=tol)
            ref.set_state(u0)
            for i in range(1, steps + 1):
                if tol == 0.0 and judge and i % judge == 0:
                    ref.advance(k)
                else:
                    nn.advance(ref, 1, k, judge_every=0)
            assert np.array_equal(one.get_state(), ref.get_state())
