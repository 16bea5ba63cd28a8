"""Layer gradients of the radiance cache where the split over sample blocks and
the sum of the blocks' partials have edges: fewer 32-sample steps than blocks, as
many, and one more, whole steps and ragged ones.  The gradients of n samples
against the mean of those of their two halves, whose loss scale is exactly twice
the whole's.  What differs is the order of a weight's n f32 terms: about
sqrt(n) 2^-24 < 4e-6 of the sum of their magnitudes, which exceeds the sum's own
norm by less than 100 on these random targets: 4e-4 of the norm."""
import numpy as np
import pytest

from tests.conftest import announce
from tests.test_cache_scatter_gpu import _samples
from voidray_amd import _native as N
from voidray_amd.device import RadianceCache

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 34, 62, 4096, 4098, 4160])
def test_layer_gradients_equal_those_of_the_halves(n, gpu_ctx):
    import torch
    cache = RadianceCache(gpu_ctx, (0, 0, 0), (1, 1, 1), log2_table=14, max_resolution=256, seed=5)
    x = _samples(torch, n, 19 + n, False)

    def gradients(s):
        out = torch.full((N.VR_CACHE_MLP_PARAMS,), 7.0, device="cuda")
        torch.cuda.synchronize()
        cache.gradients(len(s[0]), *(v.data_ptr() for v in s), d_mlp_grad=out.data_ptr())
        torch.cuda.synchronize()
        return out.cpu().numpy().astype(np.float64)

    announce(f"layer gradients of {n} samples")
    whole = gradients(x)
    halves = [gradients([v[i * n // 2:(i + 1) * n // 2].contiguous() for v in x]) for i in range(2)]
    mean = (halves[0] + halves[1]) / 2
    assert np.all(np.isfinite(whole)) and np.linalg.norm(whole) > 0
    assert np.linalg.norm(whole - mean) <= 4e-4 * np.linalg.norm(mean)
