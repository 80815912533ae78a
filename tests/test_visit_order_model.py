"""The rule by which the closest-hit loops may leave the reference's order of visits,
on a host model of them (tests/cpp/visit_order_model.cpp): random flushes and
group widths over the oracle's trees.  A ray that is no tie has the hit of a walk
in the reference's order, on scenes whose flat boxes and equal distances give other
hits under plain culling, along the axes (NaN products) and on slivers; on soups
and rooms hardly any ray is a tie.  (The kernels themselves are held to the oracle
by tests/test_gpu_visit_order.py.)
"""
import ctypes
import os
import subprocess

import numpy as np
import pytest

import oracle_py as orc
import ptamd
from test_gpu_visit_order import decals, scene, triangles

N = 4000


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    src = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "visit_order_model.cpp")
    out = str(tmp_path_factory.mktemp("model") / "visit_order_model.so")
    subprocess.run(["g++", "-std=c++17", "-O2", "-ffp-contract=off", "-Wall", "-Wextra", "-shared", "-fPIC", src, "-o", out],
                   check=True)
    lib = ctypes.CDLL(out)

    def run(tris, rays):
        b = orc.build(tris, *ptamd.scene_bounds(tris))
        s = tris[b["perm"]]
        corners = np.concatenate([s["v0"], s["v1"], s["v2"]], axis=1).astype(np.float32)
        ids, rays = s["id"].astype(np.uint32).copy(), np.ascontiguousarray(rays, np.float32)
        counts = np.zeros(7, np.uint64)
        p = [a.ctypes.data_as(ctypes.c_void_p) for a in (corners, ids, b["children"], b["bboxes"], rays, counts)]
        lib.visit_orders(len(tris), p[0], p[1], p[2], p[3], len(rays), p[4], 1, p[5])
        return [int(c) for c in counts]

    return run


@pytest.mark.parametrize("name", ["decals", "decal planes", "two tessellations", "edges", "corners", "repeated", "axes",
                                  "grazing"])
def test_flat_scenes(model, name):
    v, rays = scene(name, N)
    hits, bare_d, wrong_d, ties_d, bare_g, wrong_g, ties_g = model(triangles(v)[0], rays)
    assert hits > 0.05 * N and wrong_d == 0 and wrong_g == 0
    assert ties_d > 0 and ties_g > 0
    assert bare_g > 0 or name == "repeated"  # plain culling is not enough


def test_tilted_decals(model):
    """The same plane at an angle: boxes are thick, hits at equal distances remain."""
    a = np.linalg.qr(np.random.default_rng(9).normal(size=(3, 3)))[0].astype(np.float32)
    v, (_, rays) = decals(1500, 1, 1) @ a.T, scene("decals", N)
    rays = np.concatenate([rays[:, :3] @ a.T, rays[:, 3:] @ a.T], 1)
    hits, _, wrong_d, _, _, wrong_g, _ = model(triangles(v)[0], rays)
    assert hits > 0.05 * N and wrong_d == 0 and wrong_g == 0


@pytest.mark.parametrize("name", ["soup", "room", "room, axis planes", "slivers"])
def test_general_scenes(model, name):
    r = np.random.default_rng(4)
    d = r.normal(size=(N, 3))
    if name == "soup":
        tris, o = ptamd.gen_soup(20000, 8)[0], r.uniform(0, 1, (N, 3))
    elif name == "slivers":
        a, b, e = r.uniform(-1, 1, (4000, 3)), r.normal(size=(4000, 3)), 1e-4 * r.normal(size=(4000, 3))
        tris, o = triangles(np.stack([a, a + b, a + 0.5 * b + e], 1))[0], r.uniform(-2, 2, (N, 3))
    else:
        tris, o = ptamd.gen_sphere(100, 6, room=True)[0], r.uniform(-1.9, 1.9, (N, 3))
        if name != "room":
            d[np.arange(N), r.integers(0, 3, N)] = 0.0
    hits, _, wrong_d, ties_d, _, wrong_g, ties_g = model(tris, np.concatenate([o, d], 1))
    assert hits > 0 and wrong_d == 0 and wrong_g == 0
    assert ties_d <= 0.01 * N and ties_g <= 0.01 * N
