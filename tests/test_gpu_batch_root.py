"""Traces without scene ids in a batch of scenes go to the first scene that has
triangles, also behind empty scenes and where that scene is one triangle (it has
no root node), in every kernel they may take: one triangle, a few rays (several
lanes each), many rays with and without the root filter, counted.
"""
import numpy as np
import pytest

import oracle_py as orc
import ptamd
from ptamd import hip
from test_gpu_parity import interior_rays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("counts", [[0, 0, 40], [0, 1, 700], [1, 300], [0, 2], [0, 0, 3, 0, 50], [500, 0, 7], [0, 1], [0, 0]])
def test_trace_without_scene_ids(ctx, counts):
    print(f"[batch root] {counts}", flush=True)
    # Trees of other scenes first, so that the buffers hold their words.
    tris, infos, offs = ptamd.gen_batch(6, 2, counts=np.array([90, 800, 5, 60, 2, 900], np.uint32))
    ctx.upload_scenes(tris, offs, infos)
    tris, infos, offs = ptamd.gen_batch(len(counts), 5, counts=np.array(counts, np.uint32))
    first = next((s for s, c in enumerate(counts) if c), 0)
    for s, c in enumerate(counts):  # larger triangles in the small scenes, so that rays hit them
        if 0 < c < 100:
            for f in ("v1", "v2"):
                v = tris[offs[s]:offs[s + 1]]
                v[f] = v["v0"] + (300.0 if c < 4 else 40.0) * (v[f] - v["v0"])
    ctx.upload_scenes(tris, offs, infos)
    rays = interior_rays(3000, 7, np.zeros(3, np.float32), np.ones(3, np.float32))
    st = np.ascontiguousarray(tris[offs[first]:offs[first + 1]])
    if len(st):
        want = orc.brute(st, rays)
        assert (want[0] != ptamd.INVALID).any()
    else:
        want = (np.full(3000, ptamd.INVALID, np.uint32), np.full(3000, ptamd.FLT_MAX, np.float32),
                np.zeros((3000, 2), np.float32))
    saved = {k: ptamd.tune_get(k) for k in ("trace.blocks", "trace.filter")}
    d_rays = hip.DeviceArray.from_host(rays)
    try:
        for blocks in (2, 2048):
            for filt in (0, 1):
                ptamd.tune_set("trace.blocks", blocks)
                ptamd.tune_set("trace.filter", filt)
                for got, w in zip(ctx.trace_closest(rays), want):
                    assert np.array_equal(got.view(np.uint32), w.view(np.uint32)), (blocks, filt)
        out = [hip.DeviceArray(3000, np.uint32), hip.DeviceArray(3000, np.float32)]
        ctx.trace_closest_counted(d_rays.ptr, 3000, out[0].ptr, out[1].ptr)
        for got, w in zip(out, want):
            assert np.array_equal(got.to_host().view(np.uint32), w.view(np.uint32))
    finally:
        for k, v in saved.items():
            ptamd.tune_set(k, v)
        d_rays.free()
    assert ctx.get_status() == 0
