"""Closest-hit batches through the persistent queue at the edges of its pools and
slices (pools of 64 rays and more, a slice per 16,384 rays, at most 64): every
ray is answered once, with the bits that the grouped launch gives.
"""
import numpy as np
import pytest

import ptamd
from ptamd import hip

pytestmark = pytest.mark.gpu

KNOBS = ("trace.blocks", "trace.pool", "trace.filter")


@pytest.fixture(scope="module")
def batch(ctx):
    tris, infos = ptamd.gen_soup(3000, 4, emitter=False)
    ctx.upload_scene(tris, infos)
    rng = np.random.default_rng(8)
    n = 64 * 16384 + 4097
    rays = np.concatenate([rng.uniform(-0.5, 1.5, (n, 3)), rng.normal(size=(n, 3))], axis=1).astype(np.float32)
    return hip.DeviceArray.from_host(rays)


def trace(ctx, d_rays, n):
    ident = hip.DeviceArray.from_host(np.full(n + 64, 0xABCDABCD, np.uint32))
    t = hip.DeviceArray.from_host(np.full(n + 64, -7.0, np.float32))
    ctx.trace_closest_device(d_rays.ptr, n, ident.ptr, t.ptr, 0)
    ctx.synchronize()
    return ident.to_host(), t.to_host()


@pytest.mark.parametrize("n", [513, 16383, 32767, 32769, 100003, 64 * 16384 - 1, 64 * 16384 + 4097])
@pytest.mark.parametrize("pool", [64, 100, 4096])
@pytest.mark.parametrize("filt", [0, 1])
def test_every_ray_once(ctx, batch, n, pool, filt):
    print(f"[handout] n={n} pool={pool} filter={filt}", flush=True)
    saved = {k: ptamd.tune_get(k) for k in KNOBS}
    try:
        ptamd.tune_set("trace.blocks", 65535)
        want = trace(ctx, batch, n)
        ptamd.tune_set("trace.pool", pool)
        ptamd.tune_set("trace.filter", filt)
        for blocks in (1, 37):
            ptamd.tune_set("trace.blocks", blocks)
            got = trace(ctx, batch, n)
            np.testing.assert_array_equal(got[0], want[0])
            np.testing.assert_array_equal(got[1], want[1])
        assert (want[0][:n] != 0xABCDABCD).all() and (want[0][n:] == 0xABCDABCD).all()
    finally:
        for k, v in saved.items():
            ptamd.tune_set(k, v)
