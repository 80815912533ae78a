"""Group traversal (several lanes per ray): launches of few rays and the ends
of persistent loops give the oracle's bits, at the ray counts where the lanes
per ray change, on scenes of 0 to 3 triangles, on rays with zero direction
components and on trees deeper than the groups' LDS stacks.

`trace.blocks` sets how many lanes a launch has: with B workgroups, n rays get
2^lg lanes each for the largest lg <= 4 with n * 2^lg <= 256 * B, and lg = 0
is the persistent loop, whose last rays go on as groups."""
import sys

import numpy as np
import pytest

import oracle_py as orc
import ptamd
from test_gpu_parity import axis_rays, interior_rays

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.fixture
def knobs():
    names = ("trace.blocks", "trace.lds_stack", "trace.filter", "render.paths", "render.shade_min", "render.shade_lit",
             "render.refill")
    saved = {k: ptamd.tune_get(k) for k in names}

    def set_(**kw):
        for k, v in kw.items():
            ptamd.tune_set(k.replace("_", ".", 1), v)

    yield set_
    for k, v in saved.items():
        ptamd.tune_set(k, v)


def same(a, b):
    return np.array_equal(np.ascontiguousarray(a).view(np.uint32), np.ascontiguousarray(b).view(np.uint32))


@pytest.fixture(scope="module")
def soup():
    tris, infos = ptamd.gen_soup(3000, 8)
    bmin, bmax = ptamd.scene_bounds(tris)
    rays = np.concatenate([interior_rays(700, 1, bmin, bmax), axis_rays(300, 2, bmin, bmax),
                           ptamd.gen_shell_rays(500, 3, bmin, bmax, 1.5)])
    rays = rays[np.random.default_rng(4).permutation(len(rays))]
    o = orc.build(tris, bmin, bmax)
    return tris, infos, rays, orc.trace(tris, o, rays)


@pytest.mark.parametrize("lds", [8, 16, 32])
@pytest.mark.parametrize("filt", [0, 1])
def test_ray_counts_around_the_group_sizes(ctx, knobs, soup, lds, filt):
    tris, infos, rays, (oids, ot, ouv) = soup
    ctx.upload_scene(tris, infos)
    knobs(trace_blocks=4, trace_lds_stack=lds, trace_filter=filt)  # 1,024 lanes
    for n in (1, 3, 15, 63, 64, 65, 127, 128, 129, 255, 256, 257, 511, 512, 513, 1023, 1500):
        say(f"[group] n={n} lds={lds} filter={filt}")
        ids, t, uv = ctx.trace_closest(rays[:n])
        assert np.array_equal(ids, oids[:n]), n
        assert same(t, ot[:n]) and same(uv, ouv[:n]), n
    assert ctx.get_status() == 0


@pytest.mark.parametrize("blocks", [1, 8, 64, 512])
def test_batched_scenes_of_few_triangles(ctx, knobs, blocks):
    counts = [0, 1, 2, 3, 0, 700, 1, 65]
    tris, infos, offs = ptamd.gen_batch(len(counts), 5, counts=np.array(counts, np.uint32))
    # Large triangles in the tiny scenes, so that rays hit them.
    for s in (1, 2, 3, 6):
        for f in ("v0", "v1", "v2"):
            c = tris[f][offs[s]:offs[s + 1]]
            tris[f][offs[s]:offs[s + 1]] = 0.5 + 40.0 * (c - tris["v0"][offs[s]]) + (0.2 if f == "v2" else 0.0)
    ctx.upload_scenes(tris, offs, infos)
    rng = np.random.default_rng(6)
    n = 2000
    rays = np.concatenate([interior_rays(n - 200, 7, np.zeros(3, np.float32), np.ones(3, np.float32)),
                           axis_rays(200, 8, np.zeros(3, np.float32), np.ones(3, np.float32))])
    ids_in = rng.integers(0, len(counts) + 1, n).astype(np.uint32)  # one past the last: a miss
    want = [np.full(n, ptamd.INVALID, np.uint32), np.full(n, ptamd.FLT_MAX, np.float32), np.zeros((n, 2), np.float32)]
    for s, c in enumerate(counts):
        at = np.nonzero(ids_in == s)[0]
        if c == 0:
            continue
        st = np.ascontiguousarray(tris[offs[s]:offs[s + 1]])
        for w, got in zip(want, orc.brute(st, rays[at])):
            w[at] = got
    knobs(trace_blocks=blocks)
    say(f"[group] batched, {blocks} workgroups")
    ids, t, uv = ctx.trace_closest_scenes(rays, ids_in)
    assert np.array_equal(ids, want[0]) and same(t, want[1]) and same(uv, want[2])
    assert (ids != ptamd.INVALID).any() and ctx.get_status() == 0


@pytest.mark.parametrize("blocks", [4, 16, 32, 64, 256, 2048])
def test_deep_trees(ctx, knobs, blocks):
    """Deferred nodes beyond the groups' LDS columns (2 lanes hold 16 entries
    at the smallest setting, the tree defers 40 and more)."""
    from deep_scene import BOX_MAX, BOX_MIN, deep_rays, deep_scene

    tris, infos = deep_scene()
    ctx.upload_scene(tris, infos, BOX_MIN, BOX_MAX)
    rays = deep_rays(4096)
    oids, ot, ouv = orc.trace(tris, orc.build(tris, BOX_MIN, BOX_MAX), rays)
    for lds in (8, 16):
        say(f"[group] deep tree, {blocks} workgroups, lds={lds}")
        knobs(trace_blocks=blocks, trace_lds_stack=lds)
        ids, t, uv = ctx.trace_closest(rays)
        assert np.array_equal(ids, oids) and same(t, ot) and same(uv, ouv)
    assert ctx.get_status() == 0


@pytest.mark.parametrize("lit", [False, True])
@pytest.mark.parametrize("blocks", [2, 12, 60, 2048])
def test_frames_of_few_paths(ctx, knobs, lit, blocks):
    """47 x 31 pixels, 3 passes (4,371 paths): all lanes-per-path settings and
    the persistent loop with its groups at the end."""
    from test_oracle_lights import light

    w, h, n = 47, 31, 3
    eye, tgt = (0.5, 0.5, -1.5), (0.5, 0.5, 0.0)
    tris, infos = ptamd.gen_soup(20000, 4)
    infos["specularity"] = np.random.default_rng(1).choice(np.array([0.0, 4.0, 32.0], np.float32), len(infos))
    lights = np.array([light((1.0, 0.9, 0.8), (0.3, -1.0, 0.2), 1.5), light((0.2, 0.3, 1.0), (-0.5, -0.4, 1.0), 0.7)],
                      np.float32)[:2 if lit else 0]
    st = ptamd.Settings(4, 2, 1.0, 1)
    dirs = np.stack([ptamd.camera_corners(eye, tgt, (0, 1, 0), 60.0, w / h, *ptamd.pass_jitter(3, p, w, h))
                     for p in range(n)])
    seeds = np.arange(900, 900 + n, dtype=np.uint64)
    ctx.upload_scene(tris, infos, settings=st, lights=lights if lit else None)
    ctx.set_primary_rays(dirs[0], eye)
    b = orc.build(tris, *ptamd.scene_bounds(tris))
    o = np.zeros((h, w, 3))
    segs = 0
    for p in range(n):
        if lit:
            orc.render_pass_lit(tris, b, infos, lights, st, w, h, dirs[p], eye, p, int(seeds[p]), o)
        else:
            segs += orc.render_pass(tris, b, infos, st, w, h, dirs[p], eye, p, int(seeds[p]), o)[1]
    knobs(trace_blocks=blocks, render_paths=1)
    for lds in (8, 16):
        knobs(trace_lds_stack=lds)
        say(f"[group] frame, {blocks} workgroups, lds={lds}, lit={lit}")
        ctx.reset_frames()
        ctx.render_passes(w, h, seeds, dirs)
        rays = ctx.last_frame_rays()
        acc, spp = ctx.read_accumulator(w, h)
        assert spp == n and o.sum() > 0 and np.array_equal(acc, o)
        assert lit or rays == segs
    assert ctx.get_status() == 0


@pytest.mark.parametrize("shade,refill", [(1, 64), (7, 1), (33, 33), (64, 60)])
def test_shade_and_refill_thresholds(ctx, knobs, shade, refill):
    """Persistent frames at the edges of the batch sizes, with and without
    lights: the accumulator does not depend on them."""
    from test_oracle_lights import light

    w, h = 41, 29
    eye, tgt = (0.5, 0.5, -1.5), (0.5, 0.5, 0.0)
    tris, infos = ptamd.gen_soup(5000, 14)
    lights = np.array([light((1.0, 0.9, 0.8), (0.3, -1.0, 0.2), 1.5)], np.float32)
    st = ptamd.Settings(5, 2, 1.0, 1)
    dirs = ptamd.camera_corners(eye, tgt, (0, 1, 0), 60.0, w / h)
    b = orc.build(tris, *ptamd.scene_bounds(tris))
    knobs(trace_blocks=2, render_paths=1, render_shade_min=shade, render_shade_lit=shade, render_refill=refill)
    for lit in (False, True):
        say(f"[group] shade {shade}, refill {refill}, lit={lit}")
        ctx.upload_scene(tris, infos, settings=st, lights=lights if lit else None)
        ctx.set_primary_rays(dirs, eye)
        ctx.reset_frames()
        ctx.render_pass(w, h, 77)
        acc, _ = ctx.read_accumulator(w, h)
        o = np.zeros((h, w, 3))
        if lit:
            orc.render_pass_lit(tris, b, infos, lights, st, w, h, dirs, eye, 0, 77, o)
        else:
            orc.render_pass(tris, b, infos, st, w, h, dirs, eye, 0, 77, o)
        assert o.sum() > 0 and np.array_equal(acc, o)
    assert ctx.get_status() == 0


@pytest.mark.parametrize("blocks", [1, 64, 2048])
def test_frame_of_a_one_triangle_scene(ctx, knobs, blocks):
    tris, infos = ptamd.gen_soup(1, 3, emitter=False)
    for f, v in (("v0", (0, 0, 0)), ("v1", (1, 0, 0)), ("v2", (0, 1, 0))):
        tris[f] = np.array(v, np.float32)
    infos["emission"] = 2.0
    w, h = 16, 12
    eye = (0.3, 0.3, -1.0)
    dirs = ptamd.camera_corners(eye, (0.3, 0.3, 0.0))
    st = ptamd.Settings(2, ptamd.INVALID, 1.0, 1)
    ctx.upload_scene(tris, infos, settings=st)
    ctx.set_primary_rays(dirs, eye)
    knobs(trace_blocks=blocks, render_paths=1)
    say(f"[group] one triangle, {blocks} workgroups")
    ctx.reset_frames()
    ctx.render_pass(w, h, 5)
    acc, _ = ctx.read_accumulator(w, h)
    b = orc.build(tris, *ptamd.scene_bounds(tris))
    o, _ = orc.render_pass(tris, b, infos, st, w, h, dirs, eye, 0, 5)
    assert o.sum() > 0 and np.array_equal(acc, o)
