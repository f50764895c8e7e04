"""The work that a reconstruction program gives this framework, as cases to measure.

Every kind of case takes host arrays and returns host arrays, as the public entry points do: a controller
loads images and poses, estimates each view's depth and normal map, filters and fuses the maps, and before
all that picks each view's sources from the sparse model.  Scenes are rendered from the seed.

  view    one reference view: the problem is created from host images, run, and its maps read back
          (PatchMatchACMMCuda).  `geom` is the geometric-consistency pass, which starts from maps that an
          earlier pass left and reads the sources' depth maps; `post` adds the steps that a last pass has
          (curvature map, median filter, depth filter, mask).
  batch   many views of uneven size, source count and window together (PatchMatchBatch)
  filter  the cross-view filter of a cluster's maps, then the deduplication of the refined maps
  fusion  the fusion of a cluster's depth maps into points
  select  source views and depth ranges from the sparse model (Model)
"""
import math

import numpy as np

from sensemap_amd import abi, scene
from sensemap_amd import patch_match as pmm
from sensemap_amd.cross_filter import CrossImage, cross_filter, dedup
from sensemap_amd.fusion import FusionImage, StereoFusionOptions, fuse
from sensemap_amd.model import Model

# Pixel-iteration samples of one view that keep a drawn case below the largest listed one.
MOST_SAMPLES = 1920 * 1080 * 10 * 225 * 8


def listed():
    return [
        # a thumbnail of the coarsest pyramid level: launches and latency
        {"name": "view_160x120_n2", "kind": "view", "w": 160, "h": 120, "n": 2, "radius": 5, "step": 2,
         "iters": 5, "geom": False, "post": False, "storage": "f16", "accum": "plain", "mesh": "planes"},
        # an ordinary small view with the default window
        {"name": "view_640x480_n4", "kind": "view", "w": 640, "h": 480, "n": 4, "radius": 5, "step": 2,
         "iters": 6, "geom": False, "post": False, "storage": "f16", "accum": "plain", "mesh": "planes"},
        # odd sizes, a window without a kernel of its own, 8-bit images on the device
        {"name": "view_1021x767_n7_u8", "kind": "view", "w": 1021, "h": 767, "n": 7, "radius": 5, "step": 1,
         "iters": 3, "geom": False, "post": False, "storage": "u8", "accum": "plain", "mesh": "planes"},
        # a full-size view at high quality, the photometric pass
        {"name": "view_1920x1080_n10", "kind": "view", "w": 1920, "h": 1080, "n": 10, "radius": 7, "step": 1,
         "iters": 8, "geom": False, "post": False, "storage": "f16", "accum": "plain", "mesh": "heights"},
        # the last pass of a small view, with every step after the iterations
        {"name": "geom_640x480_n4_post", "kind": "view", "w": 640, "h": 480, "n": 4, "radius": 5, "step": 2,
         "iters": 2, "geom": True, "post": True, "storage": "f16", "accum": "plain", "mesh": "planes"},
        # the geometric pass of the full-size view
        {"name": "geom_1920x1080_n10", "kind": "view", "w": 1920, "h": 1080, "n": 10, "radius": 7, "step": 1,
         "iters": 2, "geom": True, "post": False, "storage": "f16", "accum": "plain", "mesh": "heights"},
        # a cluster's views in one batch
        {"name": "batch_12", "kind": "batch", "views": 12, "min_px": 320 * 240, "max_px": 1280 * 960,
         "n_min": 5, "n_max": 12, "iters": 4},
        # filter and deduplication of a full-size cluster
        {"name": "filter_11x1920x1080", "kind": "filter", "w": 1920, "h": 1080, "views": 11},
        # fusion of a few small maps, and of a full-size cluster
        {"name": "fusion_5x640x480", "kind": "fusion", "w": 640, "h": 480, "views": 5, "rgb": True},
        {"name": "fusion_11x1920x1080", "kind": "fusion", "w": 1920, "h": 1080, "views": 11, "rgb": False},
        # source selection for a room and for a site
        {"name": "select_60x5k", "kind": "select", "images": 60, "points": 5000, "max_num": 40, "track": 6},
        {"name": "select_500x300k", "kind": "select", "images": 500, "points": 300000, "max_num": 40, "track": 6},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["view", "view", "view", "batch", "filter", "fusion", "select"])
    if kind == "view":
        while True:
            w = _log_int(rng, 96, 1920)
            c = {"kind": "view", "w": w, "h": int(round(w * rng.uniform(0.5, 0.8))), "n": rng.randint(1, 12),
                 "radius": rng.choice([3, 4, 5, 5, 5, 6, 7, 7]), "step": rng.choice([1, 2]), "iters": rng.randint(2, 8),
                 "geom": rng.random() < 0.4, "post": False, "storage": rng.choice(["f16", "f16", "f16", "u8"]),
                 "accum": rng.choice(["plain", "plain", "plain", "compensated"]),
                 "mesh": rng.choice(["planes", "heights"])}
            c["post"] = c["geom"] and rng.random() < 0.5
            if _samples(c) <= 0.7 * MOST_SAMPLES:
                return c
    if kind == "batch":
        return {"kind": "batch", "views": rng.randint(2, 14), "min_px": 160 * 120, "max_px": _log_int(rng, 40000, 900000),
                "n_min": 2, "n_max": rng.randint(3, 12), "iters": rng.randint(2, 5)}
    if kind in ("filter", "fusion"):
        w = _log_int(rng, 120, 1700)
        c = {"kind": kind, "w": w, "h": int(round(w * rng.uniform(0.5, 0.8))), "views": rng.randint(3, 11)}
        return dict(c, rgb=rng.random() < 0.5) if kind == "fusion" else c
    images = _log_int(rng, 12, 600)
    return {"kind": "select", "images": images, "points": _log_int(rng, 500, 300000),
            "max_num": rng.randint(5, 60), "track": rng.randint(3, 9)}


def _samples(c):
    k = 2 * c["radius"] // c["step"] + 1
    return c["w"] * c["h"] * c["n"] * k * k * c["iters"]


def _rendered(c, seed, num_src):
    """A reference view and num_src sources around it, with their true depth and normal maps."""
    f = 0.8 * c["w"]
    make = scene.heightfield_scene if c.get("mesh", "heights") == "heights" else scene.planes_scene
    return make(seed=seed % 100003 + 1, width=c["w"], height=c["h"], f=f, num_src=num_src)


def _estimated(views, rng):
    """Depth and normal maps as an estimation leaves them: 0.2 percent of noise, 4 percent of outliers,
    3 percent of holes, normals a few degrees off.  The views share one field of noise, each at a shift of
    its own."""
    most_h, most_w = max(v.depth.shape[0] for v in views), max(v.depth.shape[1] for v in views)
    field = rng.standard_normal((4, most_h, most_w), dtype=np.float32)
    chance = rng.random((2, most_h, most_w), dtype=np.float32)
    maps = []
    for v in views:
        h, w = v.depth.shape
        dy, dx = int(rng.integers(0, most_h)), int(rng.integers(0, most_w))
        g, u = (np.roll(x, (dy, dx), (1, 2))[:, :h, :w] for x in (field, chance))
        d = v.depth * (1 + np.float32(0.002) * g[0])
        d[u[0] < 0.04] *= (np.float32(0.5) + u[1])[u[0] < 0.04]
        d[u[0] > 0.97] = 0
        n = v.normal + np.float32(0.05) * g[1:]
        n /= np.sqrt(n[0] * n[0] + n[1] * n[1] + n[2] * n[2]) + np.float32(1e-12)
        maps.append((d, n))
    return maps


def prepare(case, seed):
    rng = np.random.default_rng(seed)
    kind = case["kind"]
    engine = pmm.default_engine()
    if kind == "view":
        sc = _rendered(case, seed, case["n"])
        prob = scene.to_problem(sc)
        opts = pmm.PatchMatchOptions(
            window_radius=case["radius"], window_step=case["step"], sigma_spatial=float(case["radius"]),
            num_iterations=case["iters"], geom_consistency=case["geom"], thk=2, seed=seed,
            image_storage=abi.PM_STORAGE_F16 if case["storage"] == "f16" else abi.PM_STORAGE_U8,
            accum_mode=abi.PM_ACCUM_PLAIN if case["accum"] == "plain" else abi.PM_ACCUM_COMPENSATED,
            est_curvature=case["post"], median_filter=case["post"], conf_filter=case["post"])
        if case["geom"]:
            maps = _estimated([sc.ref] + sc.srcs, rng)
            prob.depth_maps = [m[0] for m in maps]
            prob.normal_maps = [m[1] for m in maps]
        if case["post"]:
            mask = np.full((case["h"], case["w"]), 255, np.uint8)
            mask[: case["h"] // 8, : case["w"] // 3] = 0
            prob.mask_maps = [mask] + [None] * case["n"]
        return {"kind": kind, "engine": engine, "options": opts, "problem": prob, "curvature": case["post"]}
    if kind == "batch":
        # sizes, sources and windows of the case; texture and random streams of the seed
        orbit = scene.orbit_scene(seed=3, num_cams=2 * case["views"] + 2, min_px=case["min_px"],
                                  max_px=case["max_px"], grid=48)
        tex = scene.Texture(orbit.texture.spacing, orbit.texture.amplitude, seed=seed % 100003 + 1)
        orbit.views = [scene.render(orbit.tris, v.camera, tex) for v in orbit.views]
        items = scene.batch_problems(orbit, num_views=case["views"], seed=3, n_min=case["n_min"],
                                     n_max=case["n_max"], iterations=case["iters"])
        for opts, _ in items:
            opts.seed = seed
        return {"kind": kind, "engine": engine, "items": items}
    if kind in ("filter", "fusion"):
        sc = _rendered(case, seed, case["views"] - 1)
        views = [sc.ref] + sc.srcs
        maps = _estimated(views, rng)
        n = len(views)
        others = [[j for j in range(n) if j != k] for k in range(n)]
        if kind == "filter":
            # the maps as NormalMap files hold them
            from sensemap_amd.io import encode_normals
            images = [CrossImage(v.camera.K, v.camera.R, v.camera.T, d, encode_normals(m))
                      for v, (d, m) in zip(views, maps)]
            return {"kind": kind, "engine": engine, "images": images, "views": list(enumerate(others))}
        images = [FusionImage(v.camera.K, v.camera.R, v.camera.T, d, m,
                              np.repeat(v.image[:, :, None], 3, axis=2) if case["rgb"] else v.image, others[k])
                  for k, (v, (d, m)) in enumerate(zip(views, maps))]
        options = StereoFusionOptions()
        pixels = case["w"] * case["h"] * n
        return {"kind": kind, "engine": engine, "images": images, "options": options, "pixels": pixels,
                "points": pixels // options.min_num_pixels}
    return {"kind": kind, "engine": engine, "model": Model(*_sparse(case, rng)),
            "max_num": min(case["max_num"], case["images"])}


def _sparse(case, rng):
    """Cameras on a jittered orbit and points inside it, each seen by a run of neighbouring cameras."""
    num, points = case["images"], case["points"]
    R = np.zeros((num, 3, 3), np.float32)
    T = np.zeros((num, 3), np.float32)
    for k in range(num):
        a = 2 * math.pi * (k + 0.4 * rng.random()) / num
        c = [12.0 * math.cos(a), -8.0 - rng.random(), 12.0 * math.sin(a)]
        R[k], T[k] = scene.look_at(c, [rng.random(), 0.0, rng.random()])
    xyz = (rng.random((points, 3)) * [16.0, 1.0, 16.0] - [8.0, 0.5, 8.0]).astype(np.float32)
    length = np.minimum(2 + rng.poisson(case["track"] - 2, points), num).astype(np.int64)
    offsets = np.concatenate([np.zeros(1, np.int64), np.cumsum(length)])
    first = rng.integers(0, num, points)
    images = (np.repeat(first - offsets[:-1], length) + np.arange(offsets[-1])) % num
    is_rig = (rng.random(num) < 0.3).astype(np.uint8)
    return R, T, xyz, offsets, images.astype(np.int32), is_rig


def _padded(a, rows):
    """`a` at the front of an array of `rows` rows, so that a case's outputs have one shape."""
    out = np.zeros((rows,) + a.shape[1:], a.dtype)
    out[: len(a)] = a
    return out


def run(state):
    kind, engine = state["kind"], state["engine"]
    if kind == "view":
        e = pmm.PatchMatchACMMCuda(state["options"], state["problem"], engine)
        e.Run()
        out = {"depth": e.GetDepthMap(), "normal": e.GetNormalMap(), "conf": e.GetConfMap()}
        if state["curvature"]:
            out["curvature"] = e.GetCurvatureMap()
        e.close()
        return out
    if kind == "batch":
        b = pmm.PatchMatchBatch(state["items"], engine)
        b.Run()
        out = [[v.GetDepthMap(), v.GetNormalMap(), v.GetConfMap()] for v in b.views]
        b.close()
        return out
    if kind == "filter":
        refined = cross_filter(state["images"], state["views"], engine=engine)
        kept = [(CrossImage(im.K, im.R, im.T, refined[k], im.normal), True) for k, im in enumerate(state["images"])]
        out = dedup(kept, state["views"], engine=engine)
        return {"refined": refined, "visibility": out["visibility"], "dedup_depth": out["dedup_depth"]}
    if kind == "fusion":
        got = fuse(state["images"], state["options"], engine)
        # a point takes at least min_num_pixels pixels, and a pixel belongs to one point
        sizes = {"vis_offsets": state["points"] + 1, "vis_images": state["pixels"]}
        return dict({k: _padded(v, sizes.get(k, state["points"])) for k, v in got.items()}, count=len(got["score"]))
    lists = state["model"].GetMaxOverlappingImages(state["max_num"], 1.0, engine=engine)
    ranges = state["model"].ComputeDepthRanges(engine=engine)
    images = np.full((len(lists), state["max_num"]), -1, np.int32)
    for row, x in zip(images, lists):
        row[: len(x)] = x
    return {"images": images, "ranges": np.array(ranges, np.float32)}


def _view_work(w, h, n, radius, step, iters, geom):
    """Images in, maps out; per pixel and iteration the ten propagated hypotheses against every source and
    the four refined ones against at least one, 23 FP32 operations per window sample and 75 around it."""
    px, k = w * h, 2 * radius // step + 1
    evals = px * iters * (10 * n + 4)
    byt = px * (1 + n + 20 + ((4 * n + 16) if geom else 0))
    return byt, evals * (23 * k * k + 75 + (61 if geom else 0))


def work(case):
    kind = case["kind"]
    if kind == "view":
        byt, flops = _view_work(case["w"], case["h"], case["n"], case["radius"], case["step"], case["iters"], case["geom"])
    elif kind == "batch":  # the mean size, source count and window of the draw
        px = (case["max_px"] - case["min_px"]) / math.log(case["max_px"] / case["min_px"])
        n = (case["n_min"] + case["n_max"]) / 2
        byt, flops = (sum(x) * case["views"] / 2 for x in zip(_view_work(px, 1, n, 5, 2, case["iters"], False),
                                                             _view_work(px, 1, n, 7, 1, case["iters"], False)))
    elif kind == "filter":  # depth and normal code in; refined and deduplicated depth, visibility out; per source
        px = case["w"] * case["h"] * case["views"]  # two projections there and back
        byt, flops = px * 20, px * (case["views"] - 1) * 120
    elif kind == "fusion":  # depth, normal and colour in; a point about every fourth pixel of one view out
        px = case["w"] * case["h"] * case["views"]
        byt, flops = px * (16 + (3 if case["rgb"] else 1)) + px / case["views"] / 4 * 60, px * (case["views"] - 1) * 60
    else:
        obs = case["points"] * case["track"]
        byt, flops = case["points"] * 20 + obs * 4 + case["images"] * (49 + 4 * case["max_num"]), obs * case["track"] * 30
    return {"bytes": byt, "flops": flops}


def tolerance(case):
    # Maps, points and lists are chosen by comparisons of computed costs, so another rounding anywhere gives
    # other choices; every kernel keeps one canonical order of FP32 operations and the same bits.
    return "exact"


def exact(case, seed):
    """The depth ranges have a 64-bit value: the camera z of the 8 corners of the box around all points and
    camera centres.  The other outputs are what comparisons chose, and have none."""
    if case["kind"] != "select":
        return None
    R, T, xyz = (np.asarray(x, np.float64) for x in _sparse(case, np.random.default_rng(seed))[:3])
    everything = np.concatenate([xyz, -np.einsum("kji,kj->ki", R, T)])
    lo, hi = everything.min(0), everything.max(0)
    corners = np.array([[x, y, z] for x in (lo[0], hi[0]) for y in (lo[1], hi[1]) for z in (lo[2], hi[2])])
    z = corners @ R[:, 2].T + T[:, 2]
    return {"images": None, "ranges": np.stack([np.maximum(z.min(0), 1e-6), z.max(0)], 1)}
