"""Frames sent while earlier ones are at work equal, bit for bit, the same calls
with a synchronisation after each: accumulators, images and ray counts, with
the calls a program makes in between (camera, seed, size, settings, scene,
rebuild, cache frames, reads), over more frames than there are slots, and at
more paths than a frame may have to be traced beside another.
"""
import numpy as np
import pytest

import ptamd
from ptamd import hip

pytestmark = pytest.mark.gpu

EYE = (0.2, 0.1, 2.5)


def corners(k, w, h):
    eye = (EYE[0] + 0.05 * k, EYE[1], EYE[2])
    return ptamd.camera_corners(eye, (0, 0, 0), (0, 1, 0), 50.0, w / h, 0.3, 0.6), eye


def scenes():
    a = ptamd.gen_soup(3000, 5)
    b = ptamd.gen_sphere(40, 9)
    return a, b


def play(ctx, calls, sync):
    """Runs the calls; returns what the reading ones saw."""
    (ta, ia), (tb, ib) = scenes()
    ctx.upload_scene(ta, ia, settings=ptamd.Settings(4, 2, 1.0, 1))
    seen = []
    images = []
    for name, *a in calls:
        if name == "frame":
            w, h, k = a
            ctx.set_primary_rays(*corners(k, w, h))
            ctx.render_pass(w, h, 100 + k)
        elif name == "frames":
            w, h, k, n = a
            d = np.stack([corners(k + j, w, h)[0] for j in range(n)])
            ctx.set_primary_rays(*corners(k, w, h))
            ctx.render_passes(w, h, np.arange(n, dtype=np.uint64) + k, d)
        elif name == "cache":
            w, h, k = a
            ctx.set_primary_rays(*corners(k, w, h))
            ctx.render_cache_frame(w, h, 7 + k, ptamd.CacheSettings(train_samples=(w * h) // 8))
        elif name == "reset":
            ctx.reset_frames()
        elif name == "settings":
            ctx.set_settings(ptamd.Settings(a[0], 1, 0.7, 1))
        elif name == "scene":
            ctx.upload_scene(tb, ib)
        elif name == "build":
            ctx.build_bvh(timed=False)
        elif name == "image":
            w, h = a
            d = hip.DeviceArray((h, w, 4), np.float32)
            ctx.read_image_device(d.ptr, w, h)
            images.append(d)
        elif name == "rays":
            seen.append(np.array([ctx.last_frame_rays()]))
        elif name == "acc":
            seen.append(ctx.read_accumulator(*a)[0])
        if sync:
            ctx.synchronize()
    ctx.synchronize()
    return seen + [d.to_host() for d in images]


PLAIN = [("frame", 97, 61, k) for k in range(9)] + [("image", 97, 61), ("rays",), ("acc", 97, 61)]
MIXED = [("frame", 64, 48, 0), ("frame", 64, 48, 1), ("image", 64, 48), ("frame", 64, 48, 2), ("reset",),
         ("frame", 64, 48, 3), ("frames", 64, 48, 4, 5), ("image", 64, 48), ("settings", 2), ("frame", 64, 48, 9),
         ("frame", 64, 48, 10), ("build",), ("frame", 64, 48, 11), ("rays",), ("frame", 64, 48, 12), ("scene",),
         ("frame", 64, 48, 13), ("frame", 64, 48, 14), ("frame", 64, 48, 15), ("image", 64, 48), ("acc", 64, 48),
         ("frame", 131, 77, 16), ("frame", 131, 77, 17), ("frames", 131, 77, 18, 20), ("frame", 131, 77, 40),
         ("image", 131, 77), ("acc", 131, 77)]
CACHED = [("frame", 80, 64, 0), ("cache", 80, 64, 1), ("frame", 80, 64, 2), ("frame", 80, 64, 3), ("rays",),
          ("cache", 80, 64, 4), ("cache", 80, 64, 5), ("frame", 80, 64, 6), ("image", 80, 64), ("acc", 80, 64)]
LARGE = [("frame", 512, 512, 0), ("frames", 512, 512, 1, 17), ("frame", 512, 512, 30), ("frames", 512, 512, 31, 2),
         ("rays",), ("acc", 512, 512)]


@pytest.mark.parametrize("name,calls", [("plain", PLAIN), ("mixed", MIXED), ("cached", CACHED), ("large", LARGE)])
def test_frames_in_flight_equal_frames_one_by_one(name, calls):
    print(f"[in flight] {name}", flush=True)
    got = []
    for sync in (True, False, False):
        ctx = ptamd.Context(0)
        ctx.cache_init(3, np.full(3, -4, np.float32), np.full(3, 4, np.float32))
        got.append(play(ctx, calls, sync))
        ctx.close()
    for k in (1, 2):
        for a, b in zip(got[0], got[k]):
            np.testing.assert_array_equal(a, b)
    assert any(np.any(a != 0) for a in got[0])
