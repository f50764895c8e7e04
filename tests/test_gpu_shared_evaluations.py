"""The sweep and local optimisation list the evaluations that a tile needs and share them among a
workgroup's waves.  Which evaluations are left out depends on the options, and the tile size on the
launch; the maps are the transcription's bit for bit in every case."""
import numpy as np
import pytest

from oracle import binding
from sensemap_amd import abi, scene
from sensemap_amd import patch_match as pmm
from tests import helpers

pytestmark = pytest.mark.gpu

CASES = {
    # more draws than a thread keeps in registers, weights by count
    "counted_draws": (dict(num_samples=37, random_optimization=False), dict()),
    "one_source": (dict(), dict(num_src=1)),
    # costs near the largest float: a zero weight need not remove them, so nothing is left out
    "unbounded_term": (dict(geom_consistency=True, geom_consistency_regularizer=1e38), dict()),
    "geometric": (dict(geom_consistency=True), dict(num_src=7)),
    # no source ever qualifies, and every source does
    "none_good": (dict(num_good_hypothesis=12), dict()),
    "all_good": (dict(num_good_hypothesis=0, num_bad_hypothesis=11), dict(num_src=6)),
    "wide_runtime_window": (dict(window_radius=9, window_step=2), dict()),
    "compensated": (dict(accum_mode=abi.PM_ACCUM_COMPENSATED, image_storage=abi.PM_STORAGE_U8), dict()),
    # a tile's last row and column, fewer pixels than a wave
    "edge": (dict(), dict(width=33, height=17)),
    "sliver": (dict(window_radius=7, window_step=1), dict(width=129, height=3)),
}


def maps(v):
    return {"depth": v.GetDepthMap(), "normal": v.GetNormalMap(), "conf": v.GetConfMap(),
            "cost": v.GetCostMap(), "view_sel": v.GetViewSelMap()}


@pytest.mark.parametrize("name", CASES)
def test_bitwise_alone_and_in_a_large_launch(name):
    options, shape = CASES[name]
    sc = scene.planes_scene(**dict(dict(seed=6, width=90, height=70, f=80.0, num_src=4), **shape))
    opts = helpers.c1_options(num_iterations=4, **options)
    prob = scene.to_problem(sc, with_gt_maps=opts.geom_consistency)
    print(f"[shared] {name}", flush=True)
    e = pmm.PatchMatchACMMCuda(opts, prob)
    e.Run()
    alone = maps(e)
    cpu = binding.run_view(opts, e.view)
    assert e.GetTile(abi.PM_PHASE_SWEEP) == e.GetTile(abi.PM_PHASE_LOCAL) == (8, 4)
    e.close()
    assert not any(helpers.maps_equal(alone, cpu).values()), helpers.maps_equal(alone, cpu)
    # alone it runs on tiles of 16 pixels; beside a larger view on tiles of 64, and beside one of more
    # tiles than the chip has workgroup slots on tiles of 256
    for width, height, tile in ((480, 320, (16, 8)), (1600, 800, (32, 16))):
        big = scene.planes_scene(seed=7, width=width, height=height, f=900.0, num_src=2)
        rest = dict(options, geom_consistency=False, num_samples=15)
        b = pmm.PatchMatchBatch([(opts, prob), (helpers.c1_options(num_iterations=4, **rest), scene.to_problem(big))])
        b.Run()
        together = maps(b.views[0])
        assert b.views[0].GetTile(abi.PM_PHASE_SWEEP) == tile
        b.close()
        assert not any(helpers.maps_equal(together, alone).values()), helpers.maps_equal(together, alone)


def test_a_counted_run_gives_the_same_maps():
    # PM_COUNT_ALL makes every evaluation of the algorithm, others leave out what cannot matter
    sc = helpers.small_heightfield()
    opts = helpers.c1_options(num_iterations=5, window_radius=7, window_step=1)
    got = []
    for counting in (False, True):
        engine = pmm.Engine(0)
        engine.set_counting(counting)
        e = pmm.PatchMatchACMMCuda(opts, scene.to_problem(sc), engine=engine)
        e.Run()
        got.append(maps(e))
        e.close()
    assert not any(helpers.maps_equal(*got).values()), helpers.maps_equal(*got)
    assert np.count_nonzero(got[0]["depth"]) > 0.9 * got[0]["depth"].size


@pytest.mark.parametrize("width,height,num_src,radius,step,sweep,local", [
    (160, 120, 4, 5, 2, (8, 4), (8, 4)),
    (320, 240, 1, 5, 2, (16, 8), (16, 8)),
    # few window samples per pixel: what a tile costs once is spread over 256 pixels
    (640, 480, 1, 5, 2, (32, 16), (32, 16)),
    (640, 480, 4, 2, 2, (32, 16), (32, 16)),
    (640, 480, 4, 5, 2, (16, 8), (32, 16)),
    (600, 450, 1, 7, 1, (16, 8), (16, 8)),
    (640, 480, 4, 7, 1, (16, 8), (16, 8)),
])
def test_tiles_follow_the_work_per_pixel(width, height, num_src, radius, step, sweep, local):
    opts = helpers.c1_options(num_iterations=4, window_radius=radius, window_step=step)
    sc = scene.planes_scene(seed=3, width=width, height=height, f=0.8 * width, num_src=num_src)
    e = pmm.PatchMatchACMMCuda(opts, scene.to_problem(sc))
    assert e.GetTile(abi.PM_PHASE_SWEEP) == (0, 0)
    print(f"[tiles] {width}x{height} sources {num_src} radius {radius}", flush=True)
    e.Run()
    got = maps(e)
    tiles = e.GetTile(abi.PM_PHASE_SWEEP), e.GetTile(abi.PM_PHASE_LOCAL)
    cpu = binding.run_view(opts, e.view)
    e.close()
    assert tiles == (sweep, local)
    assert not any(helpers.maps_equal(got, cpu).values()), helpers.maps_equal(got, cpu)


@pytest.mark.parametrize("options,num_src", [
    (dict(), 5),
    (dict(window_radius=7, window_step=1, num_samples=20, random_optimization=False), 3),
    (dict(geom_consistency=True), 4),
])
def test_counts_of_a_timed_run(options, num_src):
    opts = helpers.c1_options(num_iterations=4, **options)

    def count(view, counting, blocks_per_cu):
        engine = pmm.Engine(0)
        for phase in (abi.PM_PHASE_SWEEP, abi.PM_PHASE_LOCAL):
            engine.set_tuning(phase, opts, num_src, 5, blocks_per_cu)
        engine.set_counting(counting)
        e = pmm.PatchMatchACMMCuda(opts, view, engine=engine)
        e.Run()
        st, tiles = e.GetStats(), e.GetTile(abi.PM_PHASE_SWEEP)
        got = maps(e)
        cpu = binding.run_view(opts, e.view, count=True)
        e.close()
        engine.close()
        assert not any(helpers.maps_equal(got, cpu).values()), helpers.maps_equal(got, cpu)
        return (st.ncc_evaluations, st.ncc_samples, st.geo_evaluations), st.sweep_ncc_evaluations, tiles, cpu

    # more than 512 pixels to each of a GPU's workgroups: one source a step, the fewest evaluations
    large = scene.to_problem(scene.planes_scene(seed=4, width=450, height=310, f=360.0, num_src=num_src),
                             with_gt_maps=opts.geom_consistency)
    made, sweep, tiles, cpu = count(large, abi.PM_COUNT_MADE, 1)
    print("[counts] made", made, "all", cpu["counters"], flush=True)
    assert tiles == (32, 16)
    assert made == cpu["needed"]
    every, sweep_every, _, _ = count(large, abi.PM_COUNT_ALL, 1)
    assert every == cpu["counters"] and sweep - sweep_every == made[0] - every[0] < 0
    # several sources a step on small tiles: some more
    small = scene.to_problem(scene.planes_scene(seed=4, width=150, height=100, f=120.0, num_src=num_src),
                             with_gt_maps=opts.geom_consistency)
    made, sweep, tiles, cpu = count(small, abi.PM_COUNT_MADE, 0)
    assert tiles == (8, 4)
    assert all(n <= m for n, m in zip(cpu["needed"], made))
    assert sweep < count(small, abi.PM_COUNT_ALL, 0)[1]
