"""Closest hits where several triangles lie at the same distance or within an ulp
of it, and the boxes around them are flat: overlapping decals in one plane, two
tessellations of one wall, rays through the edges and corners of a wall's
triangles, rays along the axes, repeated triangles.  There the hit depends on
which boxes the reference's order of visits has culled, and every launch shape
-- several lanes per ray, deferred leaf tests, the ends of persistent loops, the
root filter -- has to give the reference's (the oracle's) ids, distances and
barycentrics.
"""
import numpy as np
import pytest

import oracle_py as orc
import ptamd
from ptamd import hip

pytestmark = pytest.mark.gpu

Z = 0.123
KNOBS = ("trace.blocks", "trace.lds_stack", "trace.filter", "trace.refill", "render.paths", "render.shade_min",
         "render.refill")


def triangles(v, seed=3):
    v = np.asarray(v, np.float32)
    t = np.zeros(len(v), ptamd.TRI_DTYPE)
    t["v0"], t["v1"], t["v2"] = v[:, 0], v[:, 1], v[:, 2]
    t["id"] = np.random.default_rng(seed).permutation(len(v))
    infos = np.zeros(len(v), ptamd.INFO_DTYPE)
    n = np.cross(t["v1"] - t["v0"], t["v2"] - t["v0"])
    n /= np.maximum(np.linalg.norm(n, axis=1, keepdims=True), 1e-30)
    for k in ("n0", "n1", "n2"):
        infos[k][t["id"]] = n
    infos["albedo"] = 0.7
    infos["emission"][::7] = 1.5
    return t, infos


def wall(n, axis=2, at=Z):
    """2 n^2 triangles over the square [-1, 1]^2 in the plane axis = at."""
    g = np.linspace(-1, 1, n + 1)
    a, b = np.meshgrid(np.arange(n), np.arange(n), indexing="ij")
    a, b = a.ravel(), b.ravel()
    p = [np.stack([g[a + i], g[b + j]], 1) for i, j in ((0, 0), (1, 0), (1, 1), (0, 1))]
    q = np.concatenate([np.stack([p[0], p[1], p[2]], 1), np.stack([p[0], p[2], p[3]], 1)])
    return np.insert(q, axis, at, axis=2).astype(np.float32)


def decals(n, planes, seed):
    r = np.random.default_rng(seed)
    v = r.uniform(-1, 1, (n, 1, 2)) + r.uniform(0.02, 0.4, (n, 1, 1)) * r.uniform(-1, 1, (n, 3, 2))
    z = Z + 0.37 * r.integers(0, planes, (n, 1, 1))
    return np.concatenate([v, np.broadcast_to(z, (n, 3, 1))], 2).astype(np.float32)


def rays_to(points, seed):
    """Rays through the points, from above the plane, half of them normalized."""
    r = np.random.default_rng(seed)
    n = len(points)
    o = r.uniform(-1, 1, (n, 3))
    o[:, 2] = r.uniform(1, 3, n)
    d = points - o
    k = r.random(n) < 0.5
    d[k] /= np.linalg.norm(d[k], axis=1, keepdims=True)
    return np.concatenate([o, d], 1).astype(np.float32)


def square(n, seed):
    return np.concatenate([np.random.default_rng(seed).uniform(-1, 1, (n, 2)), np.full((n, 1), Z)], 1)


def scene(name, n):
    """(triangle corners, rays)"""
    r = np.random.default_rng(11)
    if name == "decals":
        return decals(1500, 1, 1), rays_to(square(n, 2), 3)
    if name == "decal planes":
        return decals(1500, 3, 1), rays_to(square(n, 2), 3)
    if name == "two tessellations":
        return np.concatenate([wall(40), wall(27)]), rays_to(square(n, 2), 3)
    if name == "edges":
        w = wall(40)
        e, f = w[r.integers(0, len(w), n)], r.random((n, 1))
        return w, rays_to(e[:, 0] * f + e[:, 2] * (1 - f), 3)
    if name == "corners":
        w = wall(40)
        return w, rays_to(w[r.integers(0, len(w), n), 1], 3)
    if name == "repeated":
        w = wall(24)
        return np.concatenate([w, w[::2], w[::3]]), rays_to(square(n, 2), 3)
    if name == "axes":  # rays along the axes and in axis planes, many from the grid's own coordinates
        rays = np.concatenate([square(n, 5), np.zeros((n, 3))], 1)
        rays[:, 2] = 2.0
        rays[:, 5] = -1.0
        k = r.random(n) < 0.5
        rays[k, 0] = np.round(rays[k, 0] * 20) / 20
        k = r.random(n) < 0.3
        rays[k, 3] = r.normal(size=k.sum())
        return np.concatenate([wall(40), wall(27)]), rays.astype(np.float32)
    if name == "grazing":  # rays nearly in the decals' plane
        o = np.concatenate([r.uniform(-2, 2, (n, 2)), Z + 1e-6 * r.normal(size=(n, 1))], 1)
        d = np.concatenate([r.normal(size=(n, 2)), 1e-6 * r.normal(size=(n, 1))], 1)
        return decals(1500, 1, 1), np.concatenate([o, d], 1).astype(np.float32)
    raise KeyError(name)


SCENES = ["decals", "decal planes", "two tessellations", "edges", "corners", "repeated", "axes", "grazing"]


@pytest.fixture
def knobs():
    saved = {k: ptamd.tune_get(k) for k in KNOBS}

    def set_(**kw):
        for k, v in kw.items():
            ptamd.tune_set(k.replace("_", ".", 1), v)

    yield set_
    for k, v in saved.items():
        ptamd.tune_set(k, v)


def same(got, want):
    return all(np.array_equal(np.ascontiguousarray(g).view(np.uint32), np.ascontiguousarray(w).view(np.uint32))
               for g, w in zip(got, want))


@pytest.mark.parametrize("name", SCENES)
def test_hits_are_the_oracles_in_every_launch_shape(ctx, knobs, name):
    v, rays = scene(name, 20000)
    tris, infos = triangles(v)
    ctx.upload_scene(tris, infos)
    want = orc.trace(tris, orc.build(tris, *ptamd.scene_bounds(tris)), rays)
    assert (want[0] != ptamd.INVALID).mean() > 0.05
    for lds in (8, 16, 32):
        for blocks, filt, refill in ((1, 0, 48), (1, 1, 48), (37, 0, 1), (37, 1, 64), (200, 0, 48), (400, 0, 48),
                                     (2048, 0, 48)):
            print(f"[visit order] {name}, lds {lds}, {blocks} workgroups, filter {filt}, refill {refill}", flush=True)
            knobs(trace_lds_stack=lds, trace_blocks=blocks, trace_filter=filt, trace_refill=refill)
            assert same(ctx.trace_closest(rays), want), (lds, blocks, filt)
    knobs(trace_lds_stack=16, trace_blocks=2048, trace_filter=1)
    for n in (1, 63, 500, 2500, 9000):
        assert same(ctx.trace_closest(rays[:n]), [w[:n] for w in want]), n
    assert ctx.get_status() == 0


def test_hits_in_batched_scenes(ctx, knobs):
    parts = [scene(n, 4000) for n in ("decals", "edges", "axes")]
    tris = [triangles(v)[0] for v, _ in parts]
    offs = np.concatenate([[0], np.cumsum([len(t) for t in tris])]).astype(np.uint32)
    want = [np.concatenate(w) for w in zip(*[orc.trace(t, orc.build(t, *ptamd.scene_bounds(t)), r)
                                             for t, (_, r) in zip(tris, parts)])]
    infos = np.zeros(max(len(t) for t in tris), ptamd.INFO_DTYPE)
    ctx.upload_scenes(np.concatenate(tris), offs, infos)
    rays = np.concatenate([r for _, r in parts])
    ids = np.repeat(np.arange(3, dtype=np.uint32), 4000)
    mix = np.random.default_rng(1).permutation(len(rays))
    for blocks in (2, 60, 200, 2048):
        print(f"[visit order] batch, {blocks} workgroups", flush=True)
        knobs(trace_blocks=blocks)
        assert same(ctx.trace_closest_scenes(rays[mix], ids[mix]), [w[mix] for w in want]), blocks
    assert ctx.get_status() == 0


@pytest.mark.parametrize("blocks", [1, 10, 2048])
def test_frames(ctx, knobs, blocks):
    """Paths between two walls, each tessellated twice, and decals: accumulators
    equal the oracle's, in bounce levels and path by path."""
    tris, infos = triangles(np.concatenate([wall(20), wall(13), wall(20, 2, Z + 2.0), wall(9, 2, Z + 2.0), wall(12, 0, 1.0),
                                            decals(100, 1, 4)]))
    w, h, n = 61, 43, 2
    eye = (0.0, 0.0, 1.5)
    st = ptamd.Settings(4, ptamd.INVALID, 1.0, 1)
    dirs = np.stack([ptamd.camera_corners(eye, (0.05, 0.1, 0.0), (0, 1, 0), 70.0, w / h, *ptamd.pass_jitter(3, p, w, h))
                     for p in range(n)])
    seeds = np.arange(40, 40 + n, dtype=np.uint64)
    b = orc.build(tris, *ptamd.scene_bounds(tris))
    want = np.zeros((h, w, 3))
    for p in range(n):
        orc.render_pass(tris, b, infos, st, w, h, dirs[p], eye, p, int(seeds[p]), want)
    assert want.sum() > 0
    ctx.upload_scene(tris, infos, settings=st)
    ctx.set_primary_rays(dirs[0], eye)
    for paths, shade, refill in ((1, 12, 60), (1, 64, 64), (1, 1, 1), (0, 12, 60)):
        print(f"[visit order] frame, {blocks} workgroups, paths {paths}, shade {shade}, refill {refill}", flush=True)
        knobs(trace_blocks=blocks, render_paths=paths, render_shade_min=shade, render_refill=refill)
        ctx.reset_frames()
        ctx.render_passes(w, h, seeds, dirs)
        assert np.array_equal(ctx.read_accumulator(w, h)[0], want), (paths, shade, refill)
    assert ctx.get_status() == 0


def test_boxes_that_are_not_numbers(ctx, knobs):
    """A triangle whose box has a NaN bound: boxes around it are no minima and
    maxima any more, so every ray walks in the reference's order, which the
    counted trace does too.  Without such a triangle the next build is as usual."""
    v, rays = scene("two tessellations", 6000)
    bad = v.copy()
    bad[5::97, 2, 0] = np.nan
    d_rays = hip.DeviceArray.from_host(rays)
    for corners in (bad, v):
        tris, infos = triangles(corners)
        ctx.upload_scene(tris, infos, np.full(3, -1.0, np.float32), np.full(3, 1.0, np.float32))
        out = [hip.DeviceArray(len(rays), np.uint32), hip.DeviceArray(len(rays), np.float32),
               hip.DeviceArray((len(rays), 2), np.float32)]
        ctx.trace_closest_counted(d_rays.ptr, len(rays), out[0].ptr, out[1].ptr, out[2].ptr)
        want = [o.to_host() for o in out]
        assert (want[0] != ptamd.INVALID).mean() > 0.05
        for blocks, filt in ((1, 0), (1, 1), (60, 0), (2048, 0)):
            print(f"[visit order] NaN {np.isnan(corners).any()}, {blocks} workgroups, filter {filt}", flush=True)
            knobs(trace_blocks=blocks, trace_filter=filt)
            assert same(ctx.trace_closest(rays), want), (blocks, filt)
    assert ctx.get_status() == 0
