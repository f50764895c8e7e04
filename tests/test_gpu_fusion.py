"""Depth-map fusion on the device (pm_fusion_run) equals its transcription
bit for bit -- positions, normals, colours, scores, visibility and the order
of the points -- on the designed plane scenes, on an orbit of rendered views
with noisy depths, on a scene whose walks outgrow the per-walk buffers
(rerun alone with buffers for max_num_pixels), and on the 11 views of the
1920x1080 heightfield scene."""
import numpy as np
import pytest

from oracle import binding
from sensemap_amd import abi, scene
from sensemap_amd import patch_match as pmm
from sensemap_amd.fusion import FusionImage, StereoFusionOptions, fuse
from tests import test_oracle_fusion as designed

pytestmark = pytest.mark.gpu


def same(a, b):
    assert len(a["score"]) == len(b["score"]), (len(a["score"]), len(b["score"]))
    for k in ("xyz", "normal", "score"):
        x, y = a[k].view(np.uint32), b[k].view(np.uint32)
        n = int(np.sum(x != y))
        assert n == 0, (k, n)
    for k in ("rgb", "vis_offsets", "vis_images"):
        assert np.array_equal(a[k], b[k]), k


def stats(eng, images, options):
    import ctypes as C
    from sensemap_amd.fusion import FusionInputs
    inp = FusionInputs(images)
    h = C.c_void_p()
    abi.check(eng.lib.pm_fusion_run(eng.handle, C.byref(options.to_c()), len(images), inp.images, C.byref(h)))
    s = abi.pm_fusion_stats()
    abi.check(eng.lib.pm_fusion_get_stats(h, C.byref(s)))
    eng.lib.pm_fusion_destroy(h)
    return s


@pytest.mark.parametrize("case", range(7))
def test_designed_scenes(case):
    d = designed
    O = StereoFusionOptions
    cases = [
        (d.scene(), O()),
        (d.scene(), O(max_num_pixels=3, min_num_pixels=3)),
        (d.scene(depth_scale=[1, 1, 1, 1.02, 1]), O(min_num_pixels=4)),
        (d.scene(depth_scale=[1, 1, 1, 1.005, 1.008]), O()),
        (d.scene(normal_tilt=[0, 0, 15.0, 0, 0]), O(min_num_pixels=4, with_normal=False)),
        (d.scene(shifts=(0, 2, -2, 4, -3.6)), O(min_num_pixels=4, max_reproj_error=0.5)),
        (d.scene(depth_scale=[1, 1.004, 1, 1, 1], rig=[1, 0, 0, 0, 0]), O()),
    ]
    ims, o = cases[case]
    got, want = fuse(ims, o), binding.fusion(ims, o)
    print("[fusion] designed case", case, "points", len(got["score"]), flush=True)
    same(got, want)


def orbit_images(seed=8, cams=12, noise=0.002, nbr=6):
    o = scene.orbit_scene(seed=seed, num_cams=cams, min_px=120 * 90, max_px=200 * 150, grid=32, extent=20.0)
    rng = np.random.default_rng(seed)
    ims = []
    n = len(o.views)
    for k, v in enumerate(o.views):
        d = (v.depth * (1 + noise * rng.standard_normal(v.depth.shape))).astype(np.float32)
        ov = [(k + s) % n for s in (1, -1, 2, -2, 3, -3)][:nbr]
        ims.append(FusionImage(v.camera.K, v.camera.R, v.camera.T, d, v.normal, v.image, ov))
    return ims


def test_orbit_equals_transcription():
    eng = pmm.Engine(0)
    ims = orbit_images()
    for o in (StereoFusionOptions(), StereoFusionOptions(min_num_pixels=3, max_depth_error=0.02, step_size=2)):
        got, want = fuse(ims, o, eng), binding.fusion(ims, o)
        s = stats(eng, ims, o)
        print("[fusion] orbit points", len(got["score"]), "walks", s.walks, "kept", s.kept, "rounds", s.rounds,
              "alone", s.big_walks, "ms", round(s.total_ms, 2), flush=True)
        assert len(got["score"]) > 100
        same(got, want)


def test_walks_that_outgrow_their_buffers():
    # 24 cameras of one plane, 0.35 px apart, and a 4-pixel reprojection
    # bound: a walk accepts a disc of pixels in every image, more than a walk
    # graph holds, so those walks run alone
    shifts = tuple(0.35 * k for k in range(24))
    ims = designed.scene(shifts=shifts, width=64)
    o = StereoFusionOptions(max_reproj_error=4.0)
    eng = pmm.Engine(0)
    got, want = fuse(ims, o, eng), binding.fusion(ims, o)
    s = stats(eng, ims, o)
    print("[fusion] dense walks: points", len(got["score"]), "alone", s.big_walks, "rounds", s.rounds, flush=True)
    assert s.big_walks > 0
    same(got, want)


def test_full_size_eleven_views_equal_transcription():
    # the 1920x1080 heightfield scene, all 11 views fused (each overlapping the
    # other 10), depths with 0.2% noise: about 2.7 M walks over 13 dataflow
    # segments, every point bitwise equal to the transcription's
    from sensemap_amd import scene as sc_mod
    sc = sc_mod.heightfield_scene(seed=2)
    views = [sc.ref] + sc.srcs
    n = len(views)
    rng = np.random.default_rng(2)
    ims = []
    for k, v in enumerate(views):
        d = (v.depth * (1 + 0.002 * rng.standard_normal(v.depth.shape))).astype(np.float32)
        ims.append(FusionImage(v.camera.K, v.camera.R, v.camera.T, d, v.normal, v.image,
                               [j for j in range(n) if j != k]))
    o = StereoFusionOptions()
    eng = pmm.Engine(0)
    got = fuse(ims, o, eng)
    s = stats(eng, ims, o)
    print("[fusion] full size: points", len(got["score"]), "walks", s.walks, "kept", s.kept, "rounds", s.rounds,
          "chain", s.chain, "ms", round(s.total_ms, 1), flush=True)
    want = binding.fusion(ims, o)
    assert len(got["score"]) > 100000
    same(got, want)


def test_grey_and_three_channel_images_equal_transcription():
    import dataclasses
    ims = orbit_images(cams=8)
    rgb = [dataclasses.replace(im, color=np.stack([im.color] * 3, axis=-1)) for im in ims]
    o = StereoFusionOptions()
    eng = pmm.Engine(0)
    grey, col = fuse(ims, o, eng), fuse(rgb, o, eng)
    print("[fusion] grey vs three channels: points", len(grey["score"]), flush=True)
    same(grey, col)
    same(grey, binding.fusion(ims, o))


@pytest.mark.parametrize("options", [
    dict(),
    dict(max_traversal_depth=4),
    dict(max_num_pixels=7),
    dict(max_depth_error=0.2, max_reproj_error=12.0, max_normal_error=60.0),
    dict(step_size=1, min_num_pixels=2),
])
@pytest.mark.parametrize("pushes", [3, 14])
def test_replays_equal_transcription(pushes, options):
    images = orbit_images(cams=15, nbr=pushes)
    if pushes > 6:
        for k, im in enumerate(images):
            im.overlapping = [(k + s) % 15 for s in range(1, 15)]
    got, want = fuse(images, StereoFusionOptions(**options)), binding.fusion(images, StereoFusionOptions(**options))
    print("[fusion] replay", pushes, options, "points", len(got["score"]), flush=True)
    assert len(want["score"]) > 0
    same(got, want)


def one_pose_images(n, pushes, width=12, height=10):
    """n images of one pose, each overlapping the `pushes` after it: a pixel's walk reaches that pixel in
    every image and no other, so a walk from the first image has n free nodes of `pushes` free pushes each."""
    rng = np.random.default_rng(n)
    rows, cols = np.mgrid[0:height, 0:width]
    ims = []
    for k in range(n):
        depth = (10.0 * (1 + 1e-4 * rng.standard_normal((height, width)))).astype(np.float32)
        normal = (0.01 * rng.standard_normal((3, height, width))).astype(np.float32)
        normal[2] -= 1.0
        normal /= np.sqrt((normal * normal).sum(0))
        ims.append(FusionImage((100.0, (width - 1) / 2.0, 100.0, (height - 1) / 2.0), np.eye(3), np.zeros(3), depth,
                               normal, ((17 * rows + 5 * cols + k) % 200 + 20).astype(np.uint8),
                               [(k + 1 + s) % n for s in range(pushes)]))
    return ims


# A walk is replayed from registers up to 64 free nodes of up to 10 free pushes each, where no cut by depth or
# count can happen; else from the stack.  Both sides of each of the four limits.
@pytest.mark.parametrize("n,pushes,options,reached", [
    (n, pushes, {}, n) for n in (2, 63, 64, 65) for pushes in (1, 9, 10, 11) if pushes < n
] + [
    (40, 10, dict(max_traversal_depth=41), 40),
    (40, 10, dict(max_traversal_depth=40), 40),
    (40, 10, dict(max_traversal_depth=3), None),
    (40, 10, dict(max_num_pixels=40), 40),
    (40, 10, dict(max_num_pixels=39), 39),
    (64, 10, dict(max_traversal_depth=65, max_num_pixels=64), 64),
    (64, 10, dict(max_traversal_depth=64, max_num_pixels=64), 64),
])
def test_replays_at_their_limits(n, pushes, options, reached):
    images = one_pose_images(n, pushes)
    o = StereoFusionOptions(**dict(dict(min_num_pixels=2, min_num_visible_images=2), **options))
    got, want = fuse(images, o), binding.fusion(images, o)
    print("[fusion] one pose", n, pushes, options, "points", len(got["score"]), flush=True)
    if reached is not None:
        # the first image's seeds, 3 pixels inside the border, come first and take every image's pixel
        assert (np.diff(want["vis_offsets"])[:24] == reached).all()
    same(got, want)
