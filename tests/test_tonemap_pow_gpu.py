"""The tonemap's gamma pass raises a pixel's three channels together; every
channel must still be what one pow gives it, bit for bit, whatever its
neighbours are: ordinary values, zeros of both signs, negatives, denormals,
infinities and NaN mixed inside one pixel, for gammas that make the exponent
fractional, one, an integer, infinite and zero.  Mode NONE with scale 1 and
exposure 0 leaves the pow alone; the reference is the same pow routine on the
host (tests/test_f32math.py pins it).  Sizes: one pixel, a ragged image and a
clipped one."""
import numpy as np
import pytest

from tests.conftest import announce
from tests.native import f32math as F
from voidray_amd import _native as N
from voidray_amd.device import tonemap

pytestmark = pytest.mark.gpu
EDGE = np.array([0.0, -0.0, 1.0, -1.0, 1e-45, 1.1754942e-38, 1.1754944e-38, 3.4028235e38, np.inf, -np.inf, np.nan,
                 0.5, -2.0, 2.0 ** -126, 16777216.0, 0.18], np.float32)


@pytest.mark.parametrize("w,h", [(1, 1), (67, 41), (1030, 3)])
@pytest.mark.parametrize("gamma", [2.2, 1.0, 0.5, -1.0, 1e-3, 0.0, np.inf])
def test_gamma_is_one_pow_per_channel(gamma, w, h, gpu_ctx):
    rng = np.random.default_rng(w + h)
    src = np.exp(rng.uniform(-20, 12, (h, w, 4))).astype(np.float32)
    pick = rng.random((h, w, 4)) < 0.3
    src[pick] = rng.choice(EDGE, int(pick.sum()))
    announce(f"gamma pass {w}x{h}, gamma {gamma}")
    with np.errstate(divide="ignore"):
        y = np.float32(1.0) / np.float32(gamma)
    for mode in (N.VR_TONEMAP_NONE, N.VR_TONEMAP_LEGACY_NONE):
        exposure = 0.0 if mode == N.VR_TONEMAP_NONE else 1.0
        got = tonemap(gpu_ctx, src, N.vr_post_desc(w, h, 1.0, gamma, exposure, mode, 1),
                      dst=np.full_like(src, 7.0))
        x = src[:1024, :1024, :3]
        want = F.power("host", x.ravel(), np.full(x.size, y, np.float32)).reshape(x.shape)
        same = (got[:1024, :1024, :3].view(np.uint32) == want.view(np.uint32)) | \
               (np.isnan(got[:1024, :1024, :3]) & np.isnan(want))
        assert same.all(), np.argwhere(~same)[:4]


@pytest.mark.parametrize("exposure", [-140.0, -3.25, 0.0, 0.5, 7.0, 200.0])
def test_exposure_scale_is_pow_of_two(exposure, gpu_ctx):
    src = np.exp(np.random.default_rng(5).uniform(-4, 4, (9, 33, 4))).astype(np.float32)
    ex = F.power("host", np.array([2.0], np.float32), np.array([exposure], np.float32))[0]
    with np.errstate(over="ignore"):
        x = (src[..., :3] * np.float32(1.5)) * ex
    want = F.power("host", x.ravel(), np.ones(x.size, np.float32)).reshape(x.shape)
    got = tonemap(gpu_ctx, src, N.vr_post_desc(33, 9, 1.5, 1.0, exposure, N.VR_TONEMAP_NONE, 0))[..., :3]
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
