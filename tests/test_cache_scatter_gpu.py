"""Grid gradients of the radiance cache on samples that share grid entries and
on samples that do not: the gradients of n samples against the mean of those of
their two halves.  (The halves' loss scale is exactly twice the whole's, so
every rounded product is the same number or its double.)  What differs is the
order in which an entry's at most 8 n f32 terms are summed: a rounding error
of about sqrt(8 n) 2^-24 < 1.2e-5 of the sum of their magnitudes, which exceeds
the sum's own magnitude by less than 100 on these random targets: 1e-3 of the
norm per level."""
import numpy as np
import pytest

from tests.conftest import announce
from voidray_amd.device import RadianceCache

pytestmark = pytest.mark.gpu


def _samples(torch, n, seed, clustered):
    g = torch.Generator(device="cuda").manual_seed(seed)
    pos = torch.rand((n, 3), device="cuda", generator=g)
    if clustered:  # every sample in one corner of the box: the same coarse entries
        pos = pos * 0.01
    pos[: n // 8] = torch.round(pos[: n // 8])  # box corners: the last cell of every level
    unit = lambda: torch.nn.functional.normalize(torch.randn((n, 3), device="cuda", generator=g), dim=1)
    return [pos.contiguous(), unit(), unit(), torch.rand(n, device="cuda", generator=g),
            torch.rand((n, 3), device="cuda", generator=g)]


@pytest.mark.parametrize("clustered", [False, True])
@pytest.mark.parametrize("log2_table,max_res", [(14, 1024), (15, 512), (19, 1024), (19, 80), (20, 2048), (16, 40000)])
def test_gradients_equal_those_of_the_halves(log2_table, max_res, clustered, gpu_ctx):
    import torch
    cache = RadianceCache(gpu_ctx, (0, 0, 0), (1, 1, 1), log2_table=log2_table, max_resolution=max_res, seed=3)
    size = 16 * 2 * (1 << log2_table)

    def gradients(x):
        out = torch.full((size,), 7.0, device="cuda")
        torch.cuda.synchronize()
        cache.gradients(len(x[0]), *(v.data_ptr() for v in x), d_grid_grad=out.data_ptr())
        torch.cuda.synchronize()
        return out.double().cpu().numpy().reshape(16, -1)

    for n in (34, 1026, 2048, 2050, 3002, 4094):
        announce(f"grid gradients 2^{log2_table} max_res {max_res} n={n}")
        x = _samples(torch, n, n, clustered)
        whole = gradients(x)
        h = n // 2
        halves = 0.5 * (gradients([v[:h].contiguous() for v in x]) + gradients([v[h:].contiguous() for v in x]))
        for level in range(16):
            norm = np.linalg.norm(halves[level])
            assert norm > 0
            assert np.linalg.norm(whole[level] - halves[level]) <= 1e-3 * norm, (n, level)
    cache.close()
