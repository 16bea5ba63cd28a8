"""The 8-wide traversal where it can go wrong: ray origins behind t_min (whose
entry distances are negative), axis-parallel rays (zero direction components),
and trees deeper than the traversal's stack in fast memory.  Both engines walk
the same scene with the same triangle arithmetic, so the answers are equal bit
for bit."""
import numpy as np
import pytest

from tests.conftest import announce
from voidray_amd import _native as N
from voidray_amd import workloads as W
from voidray_amd.device import trace_host
from voidray_amd.scene import Materials, Mesh, Scene


def _nested(n=2000, f=0.99):
    """Triangles at x = f^k of size f^k: every box a ray from the origin enters holds all smaller ones."""
    s = f ** np.arange(n)
    p = np.stack([np.stack([s, -s, -s], 1), np.stack([s, s, -s], 1), np.stack([s, 0 * s, s], 1)], 1)
    scene = Scene.empty()
    mesh = Mesh(p.reshape(-1, 3).astype(np.float32), np.arange(3 * n, dtype=np.uint32).reshape(-1, 3))
    scene.add_object(scene.add_material(Materials.lambertian((0.5, 0.5, 0.5))), scene.add_mesh(mesh))
    return scene


def _nested_rays(n=256, seed=3):
    """Rays out of and into the tip: through the triangles and through the corners they leave open."""
    rng = np.random.default_rng(seed)
    yz = rng.uniform(-1.0, 1.0, (n, 2)).astype(np.float32)
    d = W._normalize_rows(np.concatenate([np.ones((n, 1), np.float32), yz], 1))
    o = np.zeros((n, 3), np.float32)
    back = np.arange(n) % 2 == 1
    o[back] = 2.0 * d[back]
    d[back] = -d[back]
    return o, d


def _axis_rays(n=600, seed=4):
    rng = np.random.default_rng(seed)
    o = rng.random((n, 3)).astype(np.float32)
    d = np.zeros((n, 3), np.float32)
    d[np.arange(n), np.arange(n) % 3] = np.where(np.arange(n) % 2, 1.0, -1.0)
    k = np.arange(n) % 5 == 0  # two components
    d[k, (np.arange(n)[k] + 1) % 3] = -0.0 if n % 2 else 0.6
    return o, W._normalize_rows(d)


CASES = {
    "soup": lambda: (W.random_triangle_scene(3000, seed=21), W.microbench_rays(2000, res=64)),
    "axis_parallel": lambda: (W.random_triangle_scene(3000, seed=22), _axis_rays()),
    "nested": lambda: (_nested(), _nested_rays()),
}


@pytest.mark.parametrize("t_min", [-0.5, 0.0, 1e-5, 0.25])
@pytest.mark.parametrize("case", list(CASES))
def test_wide_equals_exact_on_the_host(case, t_min):
    scene, (o, d) = CASES[case]()
    got = trace_host(scene, o, d, t_min=t_min)
    ref = trace_host(scene, o, d, t_min=t_min, engine=N.VR_ENGINE_REFERENCE)
    for k in ("prim", "t", "u", "v"):
        assert np.array_equal(got[k], ref[k]), k
    anyh = trace_host(scene, o, d, t_min=t_min, any_hit=True)["hit"]
    assert np.array_equal(anyh.astype(bool), ref["prim"] != 0xFFFFFFFF)


@pytest.mark.gpu
@pytest.mark.parametrize("case", list(CASES))
def test_wide_equals_host_on_the_gpu(case, gpu_ctx):
    scene, (o, d) = CASES[case]()
    ref = trace_host(scene, o, d, engine=N.VR_ENGINE_REFERENCE)
    announce(f"wide tree {case}")
    accel = scene.build_acceleration(gpu_ctx)
    got = accel.hit(o, d)
    for k in ("prim", "t", "u", "v"):
        assert np.array_equal(got[k], ref[k]), k
    anyh = accel.hit(o, d, any_hit=True)["hit"]
    assert np.array_equal(anyh.astype(bool), ref["prim"] != 0xFFFFFFFF)


@pytest.mark.gpu
def test_every_ray_is_fetched_once(gpu_ctx):
    """Launches of all sizes around the fetch's steps: one wave, fewer waves
    than parts, one ray a wave, a full first fetch, chunks, ragged blocks.
    Answers must be those of the same rays in one large launch (whose answers
    test_trace_gpu.py pins), and nothing beyond them is written."""
    scene = W.random_triangle_scene(2000, seed=5)
    accel = scene.build_acceleration(gpu_ctx)
    big = 1_200_001
    o, d = W.incoherent_rays(big, seed=9)
    ref = accel.hit(o, d)
    for n in (1, 2, 15, 16, 17, 63, 64, 65, 1023, 1025, 7168, 65_537, 458_751, 458_753, 1_000_003):
        announce(f"fetch n={n}")
        got = accel.hit(o[:n], d[:n])
        for k in ("prim", "t", "u", "v"):
            assert np.array_equal(got[k], ref[k][:n]), (n, k)
        anyh = accel.hit(o[:n], d[:n], any_hit=True)["hit"]
        assert np.array_equal(anyh.astype(bool), ref["prim"][:n] != 0xFFFFFFFF), n
