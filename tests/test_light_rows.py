"""Directional lights given as arrays: rows of seven floats (color, direction,
intensity), or of six with intensity 1; any other shape is refused, since the
upload reads 28 bytes a light.
"""
import numpy as np
import pytest

import ptamd

ROW = [0.9, 0.8, 0.7, 0.0, -1.0, 0.0, 1.5]


@pytest.mark.parametrize("lights,rows", [([ROW], [ROW]), (np.array([ROW, ROW], np.float64), [ROW, ROW]),
                                         (np.array([[ROW]]), [ROW]), ([ROW[:6]], [ROW[:6] + [1.0]]), ([], []),
                                         (np.zeros((0, 7)), []), (np.array([ROW, ROW])[:, ::-1], [ROW[::-1]] * 2)])
def test_rows(lights, rows):
    a = ptamd._light_rows(lights)
    assert a.dtype == np.float32 and a.shape == (len(rows), 7) and a.flags["C_CONTIGUOUS"]
    np.testing.assert_array_equal(a, np.array(rows, np.float32).reshape(-1, 7))


@pytest.mark.parametrize("shape", [(7,), (1, 5), (2, 8), (3, 1), (6,), (1, 14)])
def test_other_shapes_are_refused(shape):
    with pytest.raises(ValueError):
        ptamd._light_rows(np.ones(shape, np.float32))


@pytest.mark.gpu
def test_six_floats_render_as_intensity_one(ctx):
    """Lit cache frames and plain frames: the same bits as seven floats give, and
    light arrives."""
    tris, infos = ptamd.gen_soup(20000, 4)
    eye = (0.5, 0.5, -1.5)
    w, h = 96, 64
    dirs = ptamd.camera_corners(eye, (0.5, 0.5, 0.0), (0, 1, 0), 60.0, w / h, 0.4, 0.2)
    six = np.array([[2.0, 1.9, 1.8, 0.28, -0.94, -0.19]], np.float32)
    got = []
    for lights in (None, six, np.concatenate([six, np.ones((1, 1), np.float32)], axis=1)):
        ctx.upload_scene(tris, infos, settings=ptamd.Settings(2, 3, 1.0, 1), lights=lights)
        ctx.set_primary_rays(dirs, eye)
        ctx.cache_init(2, np.full(3, -4, np.float32), np.full(3, 4, np.float32))
        ctx.reset_frames()
        ctx.render_pass(w, h, 3)
        plain = ctx.read_accumulator(w, h)[0]
        ctx.reset_frames()
        ctx.render_cache_frame(w, h, 3, ptamd.CacheSettings(train_samples=600, train_steps=2, extra_bounces=4))
        got.append((plain, ctx.read_accumulator(w, h)[0]))
    for k in (0, 1):
        np.testing.assert_array_equal(got[1][k], got[2][k])
    assert got[1][0].sum() > got[0][0].sum()
