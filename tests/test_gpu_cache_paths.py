"""Cache frames whose training and pixel paths share one path-persistent launch
equal, bit for bit, those that trace them apart (bounce levels, and one lane
per training path): image sums, training batches, queries and ray counts.

Sizes: fewer paths than a wave's 64, a training path per pixel, so few paths
that each gets several lanes from the start, and more training paths than the
grid's waves take in one round (2,048 x 4 waves of 64).
"""
import numpy as np
import pytest

import ptamd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,samples", [(5, 3, 15), (33, 17, 561), (64, 64, 1), (200, 120, 1500),
                                         (1024, 700, 600000), (1000, 601, 0)])
@pytest.mark.parametrize("lights", [0, 1])
def test_shared_launch_equals_levels(ctx, w, h, samples, lights):
    print(f"[cache paths] {w} x {h}, {samples} training paths, {lights} lights", flush=True)
    tris, infos = ptamd.gen_sphere(24, 6)
    kw = {"lights": np.array([[0.3, -1.0, 0.2, 2.0, 1.9, 1.8]], np.float32)} if lights else {}
    ctx.upload_scene(tris, infos, settings=ptamd.Settings(1, 3, 1.0, 1), **kw)
    eye = (0.1, 0.2, 2.4)
    ctx.set_primary_rays(ptamd.camera_corners(eye, (0, 0, 0), (0, 1, 0), 60.0, w / h, 0.4, 0.2), eye)
    got = []
    try:
        for paths in (0, 1):
            ptamd.tune_set("render.paths", paths)
            ctx.cache_init(2, np.full(3, -4, np.float32), np.full(3, 4, np.float32))
            ctx.reset_frames()
            for frame in range(2):
                ctx.render_cache_frame(w, h, 5 + frame, ptamd.CacheSettings(train_samples=samples, train_steps=2,
                                                                            extra_bounces=4))
            acc = ctx.read_accumulator(w, h)[0]
            raw, pred, valid = ctx.cache_last_queries(w, h)
            got.append((acc, ctx.last_frame_rays(), ctx.cache_get_params(), valid, raw[valid], pred[valid],
                        *ctx.cache_last_batch(samples)))
    finally:
        ptamd.tune_set("render.paths", 1)
    tv = [~np.isnan(g[7][:, 0]) for g in got]
    np.testing.assert_array_equal(tv[0], tv[1])
    for k in range(6):
        np.testing.assert_array_equal(got[0][k], got[1][k])
    for k in (6, 7):
        np.testing.assert_array_equal(got[0][k][tv[0]], got[1][k][tv[1]])
