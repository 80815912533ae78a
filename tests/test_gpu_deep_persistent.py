"""Trees deeper than every LDS stack setting in the persistent closest-hit
kernels and their group tails: with few workgroups the rays outnumber the lanes,
so that no launch starts with several lanes per ray.  (Launches of few rays, which
take several lanes each, have their own test of deep trees.)  Also the queue
block that the allocation-free entry point uses again for a smaller batch.
"""
import numpy as np
import pytest

import oracle_py as orc
import ptamd
from ptamd import hip
from deep_scene import BOX_MAX, BOX_MIN, deep_rays, deep_scene

pytestmark = pytest.mark.gpu

KNOBS = ("trace.blocks", "trace.lds_stack", "trace.filter", "trace.refill")


@pytest.fixture
def knobs():
    saved = {k: ptamd.tune_get(k) for k in KNOBS}

    def set_(*values):
        for k, v in zip(KNOBS, values):
            ptamd.tune_set(k, v)

    yield set_
    for k, v in saved.items():
        ptamd.tune_set(k, v)


@pytest.fixture(scope="module")
def deep():
    tris, infos = deep_scene()
    rays = deep_rays(8192)
    want = orc.trace(tris, orc.build(tris, BOX_MIN, BOX_MAX), rays, counters=True)
    assert int(want[3][3]) >= 40
    return tris, infos, rays, want[:3]


def same(got, want):
    return all(np.array_equal(g.view(np.uint32), w.view(np.uint32)) for g, w in zip(got, want))


@pytest.mark.parametrize("lds", [8, 16, 32])
def test_stacks_that_spill(ctx, knobs, deep, lds):
    tris, infos, rays, want = deep
    ctx.upload_scene(tris, infos, BOX_MIN, BOX_MAX)
    for blocks in (1, 7, 16):  # 256 lanes each: 4,096 at most, for 8,192 rays
        for filt in (0, 1):
            for refill in (1, 48, 64):
                print(f"[deep persistent] lds {lds}, {blocks} workgroups, filter {filt}, refill {refill}", flush=True)
                knobs(blocks, lds, filt, refill)
                assert same(ctx.trace_closest(rays), want)
    assert ctx.get_status() == 0


@pytest.mark.parametrize("lds", [8, 16, 32])
def test_scenes_and_frames_that_spill(ctx, knobs, deep, lds):
    tris, infos, rays, want = deep
    offs = np.array([0, 0, len(tris)], np.uint32)
    ctx.upload_scenes(tris, offs, infos, boxes=np.concatenate([BOX_MIN, BOX_MAX] * 2))
    knobs(4, lds, 1, 48)
    print(f"[deep persistent] scene ids, lds {lds}", flush=True)
    assert same(ctx.trace_closest_scenes(rays, np.ones(len(rays), np.uint32)), want)
    # Frames from inside every box: persistent paths (4 workgroups) and bounce levels.
    w, h = 64, 40
    eye = (0.35, 0.35, 0.35)
    dirs = ptamd.camera_corners(eye, (-1.0, -0.5, -0.8), (0, 1, 0), 100.0, w / h)
    infos = infos.copy()
    infos["emission"][np.random.default_rng(3).random(len(infos)) < 0.33] = 1.0
    st = ptamd.Settings(3, ptamd.INVALID, 1.0, 1)
    ctx.upload_scene(tris, infos, BOX_MIN, BOX_MAX, settings=st)
    ctx.set_primary_rays(dirs, eye)
    o = np.zeros((h, w, 3))
    orc.render_pass(tris, orc.build(tris, BOX_MIN, BOX_MAX), infos, st, w, h, dirs, eye, 0, 9, o)
    assert o.sum() > 0
    saved = ptamd.tune_get("render.paths")
    try:
        for paths in (1, 0):
            print(f"[deep persistent] frame, lds {lds}, paths {paths}", flush=True)
            ptamd.tune_set("render.paths", paths)
            ctx.reset_frames()
            ctx.render_pass(w, h, 9)
            assert np.array_equal(ctx.read_accumulator(w, h)[0], o)
    finally:
        ptamd.tune_set("render.paths", saved)
    assert ctx.get_status() == 0


def test_noalloc_queue_block_is_used_again(ctx, knobs):
    """Two batches in a row through the static queue block, the second smaller, as
    few workgroups make both persistent."""
    tris, infos = ptamd.gen_sphere(96, 5, room=True)
    ctx.upload_scene(tris, infos)
    bmin, bmax = ptamd.scene_bounds(tris)
    knobs(64, 16, 1, 48)  # 16,384 lanes
    for n, seed in ((600000, 41), (70001, 42)):
        print(f"[deep persistent] noalloc, {n} rays", flush=True)
        rays = hip.DeviceArray.from_host(ptamd.gen_shell_rays(n, seed, bmin, bmax, 1.5))
        got = []
        for f in (ctx.trace_closest_device, ctx.trace_closest_device_noalloc):
            out = [hip.DeviceArray.from_host(np.full(n, 0xABABABAB, np.uint32)), hip.DeviceArray(n, np.float32)]
            f(rays.ptr, n, out[0].ptr, out[1].ptr, 0)
            ctx.synchronize()
            got.append([o.to_host() for o in out])
        assert same(got[0], got[1]) and not (got[0][0] == 0xABABABAB).any() and (got[0][0] != ptamd.INVALID).any()
        rays.free()
    assert ctx.get_status() == 0
