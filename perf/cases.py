"""Performance cases: the work users give this framework, through its public
entry points, from the smallest calls to the largest.

A case names a path (`path`), its sizes and options.  Scenes are the
procedural workloads of the package; like a user's program, which uploads a
scene once and queries or renders it many times, the cases of one process
share each uploaded scene.  What changes with the seed is what changes from
call to call in use: rays, random streams, images, network weights, samples.

Paths:
  trace    SceneAcceleration.trace_device: closest-hit or any-hit ray queries,
           rays and answers on the GPU
  preview  iterative_render into a host image, as an interactive viewer calls it
  render   SceneAcceleration.render_device: one pass added to an accumulator on the GPU
  serve    BatchRenderer.submit: a batch of requests over a pool of scenes
  infer    RadianceCache.infer: radiance-cache answers for given vertices
  grad     RadianceCache.gradients: forward, backward and loss of the radiance cache
  cached   RadianceCache.render_frame: a frame that queries and trains the
           cache, and the trained cache's answers at probe vertices
  tonemap  vr_tonemap_device_async: the post-processing pass
"""
import ctypes
import functools
import math

import numpy as np
import torch

from voidray_amd import _native as N
from voidray_amd import workloads as W
from voidray_amd.device import BatchRenderer, Context, RadianceCache, iterative_render, make_render_desc, scene_bounds
from voidray_amd.scene import RenderSettings

EXT = N.VR_RENDER_ENV_IS | N.VR_RENDER_RUSSIAN_ROULETTE
GRID_LEVELS = 16


def listed():
    return [
        # picking and focus queries of a viewer: one launch of a wavefront of rays
        {"name": "trace_pick", "path": "trace", "scene": "soup", "size": 10_000, "rays": 64, "coherent": 1.0,
         "any": False, "engine": "wide"},
        # the traversal benchmark: 2^20 triangles, 2^22 rays, half camera rays, half incoherent
        {"name": "trace_closest", "path": "trace", "scene": "soup", "size": 1 << 20, "rays": 1 << 22, "coherent": 0.5,
         "any": False, "engine": "wide"},
        # occlusion queries over a heightfield with spheres, a ragged count of incoherent rays
        {"name": "trace_any", "path": "trace", "scene": "terrain", "size": 224, "rays": 1_000_003, "coherent": 0.25,
         "any": True, "engine": "wide"},
        # an interactive viewer's preview of the analytic spheres demo (depth of field, HDRI), odd size
        {"name": "preview_spheres", "path": "preview", "scene": "analytic", "size": 0, "width": 161, "height": 97,
         "spp": 1, "depth": 8},
        # the cornell room of the benchmark: 512 x 512, 16 spp, depth 8
        {"name": "render_cornell", "path": "render", "scene": "cornell", "size": 0, "width": 512, "height": 512,
         "spp": 16, "depth": 8, "ext": False, "engine": "wide"},
        # a progressive pass with the reference estimator, depth 16, 2.9 M triangles
        {"name": "render_terrain_ref", "path": "render", "scene": "terrain", "size": 1024, "width": 1279,
         "height": 719, "spp": 8, "depth": 16, "ext": False, "engine": "wide"},
        # the benchmark's path-integration frame: 1080p x 64 spp, depth 16, env IS + MIS + RR
        {"name": "render_terrain", "path": "render", "scene": "terrain", "size": 1024, "width": 1920, "height": 1080,
         "spp": 64, "depth": 16, "ext": True, "engine": "wide"},
        # a progressive pass over a scene of instances, watertight triangle test
        {"name": "render_instanced", "path": "render", "scene": "instanced", "size": 256, "width": 960, "height": 540,
         "spp": 4, "depth": 16, "ext": True, "engine": "watertight"},
        # serving: a burst of requests of mixed sizes over four scenes, one batch
        {"name": "serve_batch", "path": "serve", "requests": 16, "max_spp": 8, "depth": 16},
        # radiance-cache training on the samples of a frame's training paths
        {"name": "cache_grad", "path": "grad", "samples": 1 << 16, "log2_table": 19},
        # a frame rendered with the radiance cache and its Adam steps, 960 x 540 x 4 spp
        {"name": "cached_frame", "path": "cached", "scene": "terrain", "size": 1024, "width": 960, "height": 540,
         "spp": 4, "depth": 16, "train_paths": 1 << 16, "train_steps": 8, "log2_table": 19},
        # the display pass over a 1080p accumulator
        {"name": "tonemap_1080p", "path": "tonemap", "width": 1920, "height": 1080, "mode": N.VR_TONEMAP_ACES},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    path = rng.choice(["trace", "trace", "trace", "render", "render", "render", "preview", "serve", "infer", "grad",
                       "cached", "tonemap"])
    if path == "trace":
        scene = rng.choice(["soup", "soup", "terrain", "instanced"])
        size = _log(rng, 1_000, 600_000) if scene == "soup" else _log(rng, 32, 400)
        engine = rng.choice(["wide", "wide", "wide", "watertight", "reference"])
        rays = _log(rng, 1, 1 << 22) if engine != "reference" else _log(rng, 1, 1 << 15)
        return {"path": path, "scene": scene, "size": size, "rays": rays, "coherent": round(rng.random(), 3),
                "any": rng.random() < 0.4, "engine": engine}
    if path == "preview":
        return {"path": path, "scene": rng.choice(["analytic", "cornell", "materials", "microfacet"]), "size": 0,
                "width": _log(rng, 16, 640), "height": _log(rng, 16, 480), "spp": rng.randint(1, 4),
                "depth": rng.randint(1, 16)}
    if path == "render":
        scene = rng.choice(["cornell", "materials", "microfacet", "analytic", "terrain", "terrain", "instanced"])
        size = _log(rng, 32, 400) if scene in ("terrain", "instanced") else 0
        ext = scene == "instanced" or rng.random() < 0.5
        w, h = _log(rng, 32, 1920), _log(rng, 32, 1080)
        spp = max(1, min(64, _log(rng, 1, 64), (1 << 25) // (w * h)))
        return {"path": path, "scene": scene, "size": size, "width": w, "height": h, "spp": spp,
                "depth": rng.randint(2, 16), "ext": ext,
                "engine": "watertight" if ext and rng.random() < 0.3 else "wide"}
    if path == "serve":
        return {"path": path, "requests": _log(rng, 2, 32), "max_spp": rng.randint(1, 8), "depth": rng.randint(2, 16)}
    if path in ("infer", "grad"):
        return {"path": path, "samples": _log(rng, 1, 1 << 21 if path == "infer" else 1 << 17),
                "log2_table": rng.randint(14, 19)}
    if path == "cached":
        w, h = _log(rng, 64, 960), _log(rng, 64, 540)
        return {"path": path, "scene": "terrain", "size": _log(rng, 32, 400), "width": w, "height": h,
                "spp": rng.randint(1, 4), "depth": rng.randint(4, 16), "train_paths": _log(rng, 1 << 8, 1 << 16),
                "train_steps": rng.randint(1, 8), "log2_table": rng.randint(14, 19)}
    return {"path": path, "width": _log(rng, 16, 3840), "height": _log(rng, 16, 2160),
            "mode": rng.choice([N.VR_TONEMAP_NONE, N.VR_TONEMAP_ACES, N.VR_TONEMAP_REINHARD, N.VR_TONEMAP_FILMIC,
                                N.VR_TONEMAP_UNCHARTED2])}


# ---- scenes ------------------------------------------------------------------
ENGINES = {"wide": N.VR_ENGINE_WIDE, "reference": N.VR_ENGINE_REFERENCE, "watertight": N.VR_ENGINE_WATERTIGHT}
_BUILT = {}  # (scene, size) -> (Scene, SceneAcceleration); uploaded once, as a user's program does


def _make_scene(kind, size):
    if kind == "soup":  # random triangles; from 2^20 on exactly the traversal benchmark's
        return W.random_triangle_scene(size) if size >= 1 << 20 else W.lit_random_triangle_scene(size)
    if kind == "terrain":  # the full benchmark scene at 1024, its smaller relatives below
        if size >= 1024:
            return W.terrain_spheres(grid=size)
        return W.terrain_spheres(grid=size, n_spheres=50, sphere_res=(32, 16), tex_size=512, env_size=(512, 256))
    if kind == "instanced":
        return W.terrain_spheres(grid=size, tex_size=512, env_size=(512, 256), instanced=True)
    return {"cornell": W.cornell_room, "analytic": W.analytic_spheres, "materials": W.material_spheres,
            "microfacet": W.microfacet_spheres}[kind]()


def _scene(kind, size=0):
    if (kind, size) not in _BUILT:
        small = [k for k in _BUILT if k[0] in ("soup", "terrain", "instanced") and k[1] < 1024]
        if len(small) >= 8:
            del _BUILT[small[0]]
        s = _make_scene(kind, size)
        _BUILT[(kind, size)] = (s, s.build_acceleration(Context.default()))
    return _BUILT[(kind, size)]


@functools.lru_cache(maxsize=None)
def _serving_pool():
    """Scenes of 10k to 200k triangles from both generators."""
    ctx = Context.default()
    pool = [W.lit_random_triangle_scene(10_000, seed=7), W.lit_random_triangle_scene(100_000, seed=9)]
    pool += [W.terrain_spheres(grid=g, n_spheres=ns, sphere_res=res, tex_size=512, env_size=(512, 256), seed=seed)
             for g, ns, res, seed in ((72, 20, (16, 8), 8), (224, 50, (32, 16), 10))]
    return [(s, s.build_acceleration(ctx)) for s in pool]


# ---- inputs ------------------------------------------------------------------
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFF)


def _unit(n, g):
    v = torch.randn((n, 3), device="cuda", generator=g)
    return torch.nn.functional.normalize(v, dim=1)


def _rays(case, seed):
    """`coherent` of the rays are a pinhole camera's in scanline order, the
    others start anywhere in the scene's box in any direction."""
    g = _gen(seed)
    n = case["rays"]
    nc = int(n * case["coherent"])
    if case["scene"] == "soup":
        lo, hi = (0.0, 0.0, 0.0), (1.0, 1.0, 1.0)
        eye, centre = (0.5, 0.5, -1.5), (0.5, 0.5, 0.5)
    else:
        lo, hi = (-10.0, -2.0, -10.0), (10.0, 6.0, 10.0)
        eye, centre = (0.0, 9.0, 23.0), (0.0, 0.0, 1.0)
    lo, hi, eye, centre = (torch.tensor(v, device="cuda") for v in (lo, hi, eye, centre))
    # the camera moves a little from seed to seed
    eye = eye + 0.05 * (hi - lo) * (torch.rand(3, device="cuda", generator=g) - 0.5)
    fwd = torch.nn.functional.normalize(centre - eye, dim=0)
    right = torch.nn.functional.normalize(torch.linalg.cross(fwd, torch.tensor((0.0, 1.0, 0.0), device="cuda")), dim=0)
    up = torch.linalg.cross(right, fwd)
    side = max(1, math.isqrt(max(nc - 1, 0)) + 1)
    k = torch.arange(nc, device="cuda")
    x = (2.0 * (k % side) + 1.0) / side - 1.0
    y = 1.0 - (2.0 * (k // side) + 1.0) / side
    cam = fwd + 0.4142 * (x[:, None] * right + y[:, None] * up)
    o = torch.cat([eye.expand(nc, 3), lo + (hi - lo) * torch.rand((n - nc, 3), device="cuda", generator=g)])
    d = torch.cat([torch.nn.functional.normalize(cam, dim=1), _unit(n - nc, g)])
    return o.float().contiguous(), d.float().contiguous()


def _cache_inputs(case, seed, n, lo, hi):
    """Vertices on the levels of a surface: positions in the box, unit
    directions and normals, roughness, and targets with a wide range."""
    g = _gen(seed)
    lo, hi = torch.tensor(lo, device="cuda"), torch.tensor(hi, device="cuda")
    pos = lo + (hi - lo) * torch.rand((n, 3), device="cuda", generator=g)
    pos[:, 1] = lo[1] + (hi[1] - lo[1]) * (0.5 + 0.2 * torch.sin(3.0 * pos[:, 0]) * torch.cos(2.0 * pos[:, 2]))
    rough = torch.where(torch.rand(n, device="cuda", generator=g) < 0.7, 1.0, torch.rand(n, device="cuda", generator=g))
    target = torch.exp(torch.randn((n, 3), device="cuda", generator=g) - 1.0)
    return {"pos": pos.contiguous(), "dir": _unit(n, g), "nrm": _unit(n, g), "rough": rough.contiguous(),
            "target": target.contiguous()}


def _cache_params(case, seed):
    """Weights and grid of a network that has been trained for a while."""
    g = _gen(seed ^ 0x5A5A)
    mlp = torch.cat([torch.randn(n, device="cuda", generator=g) * s for n, s in
                     ((64 * 128, 0.1), (3 * 64 * 64, 0.15), (3 * 64, 0.15))])
    mlp = torch.cat([mlp, torch.zeros(13 * 64, device="cuda")])
    grid = 0.1 * torch.randn(GRID_LEVELS * 2 * (1 << case["log2_table"]), device="cuda", generator=g)
    return mlp, grid


BOX = ((-10.0, -3.0, -10.0), (10.0, 5.0, 10.0))


def _new_cache(case, box, seed, **kw):
    cache = RadianceCache(Context.default(), *box, log2_table=case["log2_table"], max_resolution=1024, **kw)
    mlp, grid = _cache_params(case, seed)
    cache.set_params(mlp.cpu().numpy(), grid.cpu().numpy())
    return cache


def _settings(case):
    if case.get("ext"):
        return RenderSettings(total_samples=case["spp"], max_bounces=case["depth"], firefly_clamp=float("inf"))
    return RenderSettings(total_samples=case["spp"], max_bounces=case["depth"])


def prepare(case, seed):
    state = _prepare(case, seed)
    torch.cuda.synchronize()  # the library's stream does not wait for torch's
    return state


def _prepare(case, seed):
    path = case["path"]
    if path == "trace":
        _, accel = _scene(case["scene"], case["size"])
        o, d = _rays(case, seed)
        n = case["rays"]
        out = ({"hit": torch.zeros(n, dtype=torch.uint8, device="cuda")} if case["any"] else
               {"prim": torch.zeros(n, dtype=torch.int32, device="cuda"),
                **{k: torch.zeros(n, device="cuda") for k in "tuv"}})
        return {"case": case, "accel": accel, "o": o, "d": d, "out": out}
    if path == "preview":
        _, accel = _scene(case["scene"])
        return {"case": case, "accel": accel, "seed": seed, "settings": _settings(case),
                "image": np.zeros((case["height"], case["width"], 4), np.float32)}
    if path == "render":
        _, accel = _scene(case["scene"], case["size"])
        st = _settings(case)
        flags = N.VR_RENDER_ALPHA_PER_CALL | (EXT if case["ext"] else 0)
        desc = make_render_desc(case["width"], case["height"], case["spp"], case["spp"], st, seed=seed, flags=flags,
                                rr_depth=4, engine=ENGINES[case["engine"]])
        return {"case": case, "accel": accel, "desc": desc,
                "image": torch.zeros((case["height"], case["width"], 4), device="cuda")}
    if path == "serve":
        pool = _serving_pool()
        rng = np.random.default_rng([seed, case["requests"]])
        # every request is a frame of its own: its image is stored, not added
        flags = N.VR_RENDER_ALPHA_PER_CALL | N.VR_RENDER_OVERWRITE | EXT
        images, requests = [], []
        for i in range(case["requests"]):
            # sizes and scenes belong to the case, streams to the seed
            w, h = W.SERVING_RESOLUTIONS[(5 * i) % 3]
            spp = 1 + (7 * i + 3) % case["max_spp"]
            st = RenderSettings(total_samples=spp, max_bounces=case["depth"], firefly_clamp=float("inf"))
            images.append(torch.zeros((h, w, 4), device="cuda"))
            requests.append((pool[i % len(pool)][1],
                             make_render_desc(w, h, spp, spp, st, seed=int(rng.integers(1 << 40)), request=i,
                                              flags=flags, rr_depth=4), images[-1].data_ptr()))
        return {"case": case, "batch": BatchRenderer(Context.default()), "requests": requests, "images": images}
    if path in ("infer", "grad"):
        n = case["samples"]
        s = {"case": case, "cache": _new_cache(case, BOX, seed), "in": _cache_inputs(case, seed, n, *BOX)}
        if path == "infer":
            s["out"] = torch.zeros((n, 3), device="cuda")
        else:
            s["out"] = {"mlp": torch.zeros(N.VR_CACHE_MLP_PARAMS, device="cuda"),
                        "grid": torch.zeros(GRID_LEVELS * 2 * (1 << case["log2_table"]), device="cuda"),
                        "loss": torch.zeros(1, device="cuda")}
        return s
    if path == "cached":
        scene, accel = _scene(case["scene"], case["size"])
        lo, hi = scene_bounds(scene)
        box = (lo.tolist(), hi.tolist())
        st = RenderSettings(total_samples=case["spp"], max_bounces=case["depth"], firefly_clamp=float("inf"))
        desc = make_render_desc(case["width"], case["height"], case["spp"], case["spp"], st, seed=seed,
                                flags=N.VR_RENDER_ALPHA_PER_CALL | EXT, rr_depth=4)
        probes = 4096
        return {"case": case, "accel": accel, "desc": desc, "cache": _new_cache(case, box, seed, lr_grid=2e-3),
                "frame": 0,
                "image": torch.zeros((case["height"], case["width"], 4), device="cuda"),
                "in": _cache_inputs(case, seed, probes, *box), "probe": torch.zeros((probes, 3), device="cuda")}
    if path == "tonemap":
        g = _gen(seed)
        src = torch.rand((case["height"], case["width"], 4), device="cuda", generator=g) ** 3 * 8.0
        src[..., 3] = 1.0
        post = N.vr_post_desc(case["width"], case["height"], 1.25, 2.2, 0.5, case["mode"], 0)
        return {"case": case, "src": src.contiguous(), "dst": torch.zeros_like(src), "post": post}
    raise ValueError(path)


def run(state):
    case = state["case"]
    path = case["path"]
    if path == "trace":
        out = state["out"]
        ptr = {"d_" + k: v.data_ptr() for k, v in out.items()}
        state["accel"].trace_device(state["o"].data_ptr(), state["d"].data_ptr(), case["rays"], any_hit=case["any"],
                                    engine=ENGINES[case["engine"]], **ptr)
        return out
    if path == "preview":
        iterative_render(state["image"], state["accel"], state["settings"], case["spp"], seed=state["seed"],
                         flags=N.VR_RENDER_ALPHA_PER_CALL)
        return state["image"]
    if path == "render":
        state["accel"].render_device(state["image"].data_ptr(), state["desc"])
        return state["image"]
    if path == "serve":
        state["batch"].submit(state["requests"], shortest_first=True)
        return state["images"]
    i = state.get("in")
    if path == "infer":
        state["cache"].infer(case["samples"], i["pos"].data_ptr(), i["dir"].data_ptr(), i["nrm"].data_ptr(),
                             i["rough"].data_ptr(), state["out"].data_ptr())
        return state["out"]
    if path == "grad":
        o = state["out"]
        state["cache"].gradients(case["samples"], i["pos"].data_ptr(), i["dir"].data_ptr(), i["nrm"].data_ptr(),
                                 i["rough"].data_ptr(), i["target"].data_ptr(), o["mlp"].data_ptr(),
                                 o["grid"].data_ptr(), o["loss"].data_ptr())
        return o
    if path == "cached":
        state["cache"].render_frame(state["accel"], state["image"].data_ptr(), state["desc"],
                                    train_paths=case["train_paths"], train_vertices=4, cache_depth=2,
                                    train_steps=case["train_steps"], frame=state["frame"], query_roughness=0.3)
        state["frame"] += 1
        # a viewer's look at what the cache holds now
        state["cache"].infer(len(state["probe"]), i["pos"].data_ptr(), i["dir"].data_ptr(), i["nrm"].data_ptr(),
                             i["rough"].data_ptr(), state["probe"].data_ptr())
        return {"image": state["image"], "probe": state["probe"]}
    post = state["post"]
    N.check(N.lib().vr_tonemap_device_async(Context.default().handle, ctypes.byref(post), state["src"].data_ptr(),
                                            state["dst"].data_ptr(), None))
    return state["dst"]


# ---- what a pass cannot do without ------------------------------------------------
MLP_FLOPS = 2 * (128 * 64 + 3 * 64 * 64 + 64 * 16)
# vertices of a path, in the scenes' own depth limits: escapes and roulette end paths early
PATH_VERTICES = 3.0
SEGMENT_FLOPS = 600.0  # a few tree nodes, a triangle test and a material per segment


def _path_work(paths, pixels):
    # paths live on the chip in the best case: per pixel the target is read and written
    return {"bytes": 32.0 * pixels, "flops": paths * PATH_VERTICES * SEGMENT_FLOPS}


def _grid_bytes(case, n):
    """Grid entries a pass over n samples reads: 8 corners of 4 bytes a level, no more than the table."""
    return GRID_LEVELS * 4.0 * min(8 * n, 1 << case["log2_table"])


def work(case):
    path = case["path"]
    if path == "trace":
        n = case["rays"]
        # rays in and answers out; the tree walked needs log(size) boxes and a triangle per ray
        return {"bytes": n * (25.0 if case["any"] else 40.0), "flops": n * SEGMENT_FLOPS}
    if path in ("preview", "render"):
        px = case["width"] * case["height"]
        return _path_work(px * case["spp"], px)
    if path == "serve":
        px = paths = 0
        for i in range(case["requests"]):
            w, h = W.SERVING_RESOLUTIONS[(5 * i) % 3]
            px += w * h
            paths += w * h * (1 + (7 * i + 3) % case["max_spp"])
        return _path_work(paths, px)
    if path == "infer":
        n = case["samples"]
        return {"bytes": n * 52.0 + _grid_bytes(case, n), "flops": float(n) * MLP_FLOPS}
    if path == "grad":
        n = case["samples"]
        return {"bytes": n * 52.0 + _grid_bytes(case, n) + 4.0 * GRID_LEVELS * 2 * (1 << case["log2_table"]),
                "flops": 3.0 * n * MLP_FLOPS}
    if path == "cached":
        px = case["width"] * case["height"]
        paths = px * case["spp"]
        w = _path_work(paths, px)
        samples = min(case["train_paths"], paths) * 3.0
        return {"bytes": w["bytes"] + paths * 52.0 + 2 * samples * 52.0,
                "flops": w["flops"] + paths * MLP_FLOPS + 3.0 * samples * MLP_FLOPS}
    px = case["width"] * case["height"]
    return {"bytes": 32.0 * px, "flops": 100.0 * px}


# ---- the same in 64 bits ------------------------------------------------------------
def _exact_trace(case, seed):
    """Moeller-Trumbore of every ray against every triangle, determinant
    threshold t_min, smallest t; small triangle soups only."""
    if case["scene"] != "soup" or case["size"] * case["rays"] > 5e9 or case["size"] > 200_000:
        return None
    if case["any"] or case["engine"] == "watertight":
        return None
    scene = _make_scene(case["scene"], case["size"])
    tri = torch.cat([torch.from_numpy(m.positions[m.indices.reshape(-1).astype(np.int64)].reshape(-1, 3, 3))
                     for m in scene.meshes]).cuda().double()
    o, d = (x.double() for x in _rays(case, seed))
    p0, e1, e2 = tri[:, 0], tri[:, 1] - tri[:, 0], tri[:, 2] - tri[:, 0]
    best = {k: torch.zeros(len(o), dtype=torch.float64, device="cuda") for k in "tuv"}
    step = max(1, 20_000_000 // len(tri))
    for a in range(0, len(o), step):
        oo, dd = o[a:a + step, None], d[a:a + step, None]
        h = torch.linalg.cross(dd.expand(-1, len(tri), 3), e2.expand(len(oo), -1, 3))
        det = (e1 * h).sum(-1)
        f = 1.0 / det
        s = oo - p0
        u = f * (s * h).sum(-1)
        q = torch.linalg.cross(s, e1.expand(len(oo), -1, 3))
        v = f * (dd * q).sum(-1)
        t = f * (e2 * q).sum(-1)
        ok = (det.abs() >= 1e-5) & (u >= 0) & (u <= 1) & (v >= 0) & (u + v <= 1) & (t > 1e-5)
        t = torch.where(ok, t, math.inf)
        m, at = t.min(1)
        hit = m < math.inf
        for k, x in (("t", t), ("u", u), ("v", v)):
            best[k][a:a + step] = torch.where(hit, x.gather(1, at[:, None])[:, 0], 0.0)
    return {"prim": None, **best}


def _resolutions():
    b = math.exp((math.log(1024.0) - math.log(16.0)) / (GRID_LEVELS - 1))
    return [int(math.floor(16.0 * b ** l + 1e-6)) for l in range(GRID_LEVELS)]


def _exact_network(case, seed, train):
    """Hash grid, one-blob encodings and MLP in 64 bits with the forward
    parameters (FP16 grid, BF16 weights), and the gradients of the mean
    relative L2 loss whose denominator is held constant."""
    n = case["samples"]
    mlp, grid = _cache_params(case, seed)
    grid = grid.half().double().reshape(GRID_LEVELS, 1 << case["log2_table"], 2).requires_grad_(train)
    mlp = mlp.bfloat16().double().requires_grad_(train)
    x = {k: v.double() for k, v in _cache_inputs(case, seed, n, *BOX).items()}
    lo, hi = (torch.tensor(v, device="cuda", dtype=torch.float64) for v in BOX)
    p = ((x["pos"] - lo) / (hi - lo).max()).clamp(0.0, 1.0)
    table = 1 << case["log2_table"]
    feats = []
    for l, r in enumerate(_resolutions()):
        g = p * r
        c = g.floor().clamp(max=r - 1).long()
        f = g - c
        acc = 0.0
        for k in range(8):
            off = torch.tensor([k & 1, (k >> 1) & 1, (k >> 2) & 1], device="cuda")
            xyz = c + off
            if (r + 1) ** 3 <= table:
                i = xyz[:, 0] + (r + 1) * (xyz[:, 1] + (r + 1) * xyz[:, 2])
            else:
                i = (xyz[:, 0] ^ ((xyz[:, 1] * 2654435761) & 0xFFFFFFFF) ^ ((xyz[:, 2] * 805459861) & 0xFFFFFFFF))
                i = i & (table - 1)
            wgt = torch.where(off.bool(), f, 1.0 - f).prod(1)
            acc = acc + wgt[:, None] * grid[l][i]
        feats.append(acc)

    def blob(v, bins):
        b = torch.arange(bins, device="cuda", dtype=torch.float64) + 0.5
        return torch.exp(-0.5 * (v[:, None] * bins - b) ** 2)

    for v in (x["dir"], x["nrm"]):
        feats.append(blob(torch.acos(v[:, 1].clamp(-1.0, 1.0)) / math.pi, 16))
        feats.append(blob(torch.atan2(v[:, 2], v[:, 0]) / (2.0 * math.pi) + 0.5, 16))
    feats.append(blob(x["rough"].clamp(0.0, 1.0), 8))
    feats.append(torch.ones((n, 1), device="cuda", dtype=torch.float64))
    feats.append(torch.zeros((n, 23), device="cuda", dtype=torch.float64))
    h = torch.cat(feats, 1)
    at = 0
    for rows, cols in ((64, 128), (64, 64), (64, 64), (64, 64), (16, 64)):
        h = h @ mlp[at:at + rows * cols].reshape(rows, cols).T
        at += rows * cols
        if rows == 64:
            h = h.relu()
    y = h[:, :3]
    if not train:
        return y
    loss = ((y - x["target"]) ** 2 / (y.detach() ** 2 + 0.01)).sum() / (3.0 * n)
    loss.backward()
    return {"mlp": mlp.grad, "grid": grid.grad.reshape(-1), "loss": loss.detach().reshape(1)}


def _exact_tonemap(case, seed):
    state = prepare(case, seed)
    c = state["src"].double()[..., :3] * 1.25 * 2.0 ** 0.5
    mode = case["mode"]
    if mode == N.VR_TONEMAP_ACES:
        a = torch.tensor([[0.59719, 0.35458, 0.04823], [0.076, 0.90834, 0.01566], [0.0284, 0.13383, 0.83777]],
                         device="cuda", dtype=torch.float64)
        b = torch.tensor([[1.60475, -0.53108, -0.07367], [-0.10208, 1.10813, -0.00605], [-0.00327, -0.07276, 1.07602]],
                         device="cuda", dtype=torch.float64)
        c = c @ a.T
        c = (c * (c + 0.0245786) - 0.000090537) / (c * (0.983729 * c + 0.432951) + 0.238081)
        c = c @ b.T
    elif mode == N.VR_TONEMAP_REINHARD:
        luma = (c * torch.tensor([0.2126, 0.7152, 0.0722], device="cuda", dtype=torch.float64)).sum(-1, keepdim=True)
        c = c * (luma * (1.0 + luma / 4.0) / (1.0 + luma) / luma)
    elif mode == N.VR_TONEMAP_FILMIC:
        c = (c - 0.004).clamp(min=0.0)
        c = (c * (6.2 * c + 0.5)) / (c * (6.2 * c + 1.7) + 0.06)
    elif mode == N.VR_TONEMAP_UNCHARTED2:
        def curve(v):
            return (v * (0.15 * v + 0.05) + 0.004) / (v * (0.15 * v + 0.5) + 0.06) - 0.02 / 0.3
        c = curve(2.0 * c) / curve(torch.tensor(11.2, dtype=torch.float64))
    gamma = float(np.float32(2.2))
    return torch.cat([c ** (1.0 / gamma), torch.ones_like(c[..., :1])], -1)


def exact(case, seed):
    path = case["path"]
    if path == "trace":
        return _exact_trace(case, seed)
    if path in ("infer", "grad"):
        return _exact_network(case, seed, path == "grad")
    if path == "tonemap":
        return _exact_tonemap(case, seed)
    return None  # a path tracer's image has no value in 64 bits on the same decisions
