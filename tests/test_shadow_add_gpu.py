"""Next-event terms are added to a path's radiance where a shadow ray's result
is written: by the wide any-hit kernel, or by the exact engine's kernel for the
rays it traces.  Both engines answer every query alike, so an extended render
must come out the same, bit for bit, and count the same segments: one ray (a
group of lanes to a ray), a ragged image whose late bounces thin out to
nothing, and one with the deepest path limit."""
import numpy as np
import pytest

from tests.conftest import announce
from tests.test_render_extended_gpu import EXT, flat_scene, small_terrain
from voidray_amd import _native as N
from voidray_amd.device import make_render_desc
from voidray_amd.scene import RenderSettings

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("scene,w,h,spp,depth", [("terrain", 1, 1, 1, 4), ("terrain", 97, 61, 3, 16),
                                                 ("flat", 65, 33, 2, 64)])
def test_both_writers_add_the_same_terms(scene, w, h, spp, depth, gpu_ctx):
    acc = (small_terrain() if scene == "terrain" else flat_scene()).build_acceleration(gpu_ctx)
    out = []
    for engine in (N.VR_ENGINE_WIDE, N.VR_ENGINE_REFERENCE):
        announce(f"shadow terms: {scene} {w}x{h}x{spp}, depth {depth}, engine {engine}")
        img = np.zeros((h, w, 4), np.float32)
        settings = RenderSettings(firefly_clamp=float("inf"), max_bounces=depth)
        desc = make_render_desc(w, h, spp, spp, settings, seed=11, request=3, flags=EXT, rr_depth=4, engine=engine)
        st = acc.render(img, desc)
        out.append((img, st["segments"], st["samples"], st["env_misses"]))
    assert out[0][1:] == out[1][1:]
    assert np.array_equal(out[0][0].view(np.uint32), out[1][0].view(np.uint32))
