"""Bottom-up tree build at the edges of its blocks (1,024 leaves) and levels (16
blocks): the parity arrays equal the oracle's, for spread and for equal keys
and for batches whose scenes begin, end and cross anywhere in a block."""
import sys

import numpy as np
import pytest

import oracle_py as orc
import ptamd
from test_gpu_parity import check_build, soup_dups

pytestmark = pytest.mark.gpu


def say(*a):
    print(*a, flush=True)
    sys.stdout.flush()


@pytest.mark.parametrize("n", [2, 1023, 1024, 1025, 2047, 2048, 2049, 16383, 16384, 16385, 262145])
@pytest.mark.parametrize("keys", ["spread", "equal", "line"])
def test_block_and_level_edges(ctx, n, keys):
    if keys == "equal":
        tris, infos = soup_dups(n)
    else:
        tris, infos = ptamd.gen_soup(n, 41, emitter=False)
        if keys == "line":  # centroids on one axis: long common prefixes, uneven trees
            for f in ("v0", "v1", "v2"):
                tris[f][:, 1:] = 0.001 * tris[f][:, 1:]
                tris[f][:, 0] = tris[f][:, 0] ** 8
    check_build(ctx, tris, infos, tag=f"{keys} {n}")
    assert ctx.get_status() == 0
    if keys != "equal":
        ctx.verify_bvh()


@pytest.mark.parametrize("seed", [0, 1, 2])
def test_batches_across_blocks(ctx, seed):
    rng = np.random.default_rng(seed)
    counts = rng.choice([0, 1, 2, 3, 100, 1023, 1024, 1025, 3000, 20000], 40).astype(np.uint32)
    tris, infos, offs = ptamd.gen_batch(len(counts), 9 + seed, counts=counts)
    say(f"[tree] batch of {len(counts)} scenes, {len(tris)} triangles")
    ctx.upload_scenes(tris, offs, infos)
    for s, c in enumerate(counts):
        if c == 0:
            continue
        t = np.ascontiguousarray(tris[offs[s]:offs[s + 1]])
        g = ctx.get_bvh_scene(s)
        o = orc.build(t, *ptamd.scene_bounds(t))
        for k in g:
            assert np.array_equal(g[k].view(np.uint32), o[k].view(np.uint32)), (s, int(c), k)
    assert ctx.verify_bvh() == 0 and ctx.get_status() == 0
