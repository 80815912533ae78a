"""The build's sort with each scene as a segment of its own, with scene passes
(many small scenes) and on one scene: the batch's trees equal, bit for bit, the
trees of its scenes uploaded alone.

Sizes sit at the edges of a 4,096-key tile and of the 32 tiles up to which a
segment's scatter adds up its tiles' counts without a scan launch.
"""
import numpy as np
import pytest

import ptamd

pytestmark = pytest.mark.gpu

TILE, FEW = 4096, 32
MIXES = {
    "one tile": [2, 3, TILE],
    "tile edges": [TILE - 1, 0, TILE + 1, 1, 2 * TILE, 0],
    "scan edges": [FEW * TILE, 5, FEW * TILE + 1, TILE, (FEW + 1) * TILE + 7],
    "several scans": [0, (FEW + 1) * TILE, 1, (FEW + 9) * TILE + 3, (FEW + 2) * TILE],
    "small scenes as segments": [3 + k % 9 for k in range(1200)],
    "scene passes": [1 + k % 13 for k in range(1700)] + [FEW * TILE // 16],
    "scene passes, scanned": [k % 5 for k in range(4000)] + [(FEW + 1) * TILE + 5] + [2] * 300,
}


@pytest.mark.parametrize("name", list(MIXES))
def test_batch_equals_scenes_alone(name):
    counts = MIXES[name]
    print(f"[segments] {name}", flush=True)
    tris, infos = ptamd.gen_soup(sum(counts), 21, emitter=False)
    # Coarse coordinates in part of the triangles: equal keys, order by index.
    verts = tris.view(np.float32).reshape(len(tris), -1)[:, :9]
    verts[::3] = np.round(verts[::3] * 4) / 4
    offs = np.concatenate([[0], np.cumsum(counts)]).astype(np.uint32)
    batch, alone = ptamd.Context(0), ptamd.Context(0)
    try:
        batch.upload_scenes(tris, offs, infos)
        batch.build_bvh()  # a second build: the buffers have been swapped
        pick = [k for k in range(len(counts)) if counts[k] > 0]
        if len(pick) > 40:
            pick = pick[:12] + pick[len(pick) // 2: len(pick) // 2 + 12] + pick[-12:]
            pick.append(int(np.argmax(counts)))
        for k in pick:
            got = batch.get_bvh_scene(k)
            alone.upload_scenes(tris[offs[k]:offs[k + 1]], np.array([0, counts[k]], np.uint32), infos)
            want = alone.get_bvh_scene(0)
            for field in want:
                np.testing.assert_array_equal(got[field], want[field], err_msg=f"scene {k}: {field}")
            order = want["perm"][np.argsort(want["perm"], kind="stable")]
            np.testing.assert_array_equal(order, np.arange(counts[k], dtype=np.uint32))
            keys, perm = got["morton"].astype(np.int64), got["perm"].astype(np.int64)
            assert (np.diff(keys) >= 0).all()
            assert (np.diff(perm)[np.diff(keys) == 0] > 0).all()
    finally:
        batch.close()
        alone.close()
