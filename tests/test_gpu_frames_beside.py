"""Frames that are traced beside the one before them: that they are (the library
counts them), that more of them than there are slots, with lights, surface
detail, a screen buffer, other streams and growing sizes, give the bits of frames
one by one, and that a frame's reported time is the frame's, not what is left of
it once the frame before has ended.

A long frame goes first, so that the next ones find it at work; cameras are made
before the first call.
"""
import numpy as np
import pytest

import ptamd
from ptamd import hip
from test_gpu_render import random_detail
from test_oracle_lights import light

pytestmark = pytest.mark.gpu

EYE = (0.5, 0.5, -1.5)
SLOTS = 3


def camera(w, h, k):
    return ptamd.camera_corners(EYE, (0.5, 0.5, 0.0), (0, 1, 0), 55.0 + k, w / h, 0.3, 0.6)


@pytest.fixture
def own():
    c = ptamd.Context(0)
    yield c
    c.close()


def beside():
    return ptamd.tune_get("render.beside")


def play(c, sizes, sync, screen=None):
    """A long frame, then one frame of each size (the accumulator restarts where
    the size changes); the accumulators of the last size."""
    cams = [camera(w, h, k % 5) for k, (w, h) in enumerate(sizes)]
    w, h = sizes[0]
    seeds = np.arange(64, dtype=np.uint64)
    many = np.stack([camera(w, h, k % 5) for k in range(64)])
    c.synchronize()
    c.set_primary_rays(cams[0], EYE)
    c.reset_frames()
    c.render_passes(w, h, seeds, many)
    if sync:
        c.synchronize()
    for k, (w, h) in enumerate(sizes):
        c.set_primary_rays(cams[k], EYE)
        c.render_pass(w, h, 1000 + k)
        if sync:
            c.synchronize()
    w, h = sizes[-1]
    acc, spp = c.read_accumulator(w, h)
    return acc, spp, c.last_frame_rays()


@pytest.mark.parametrize("sizes", [[(200, 150)] * 9, [(97, 61)] * 4 + [(160, 120)] * 4 + [(320, 200)] * 5 + [(64, 48)] * 4])
@pytest.mark.parametrize("look", ["plain", "lights", "detail"])
def test_more_frames_than_slots(own, sizes, look):
    print(f"[beside] {look}, {len(sizes)} frames", flush=True)
    tris, infos = ptamd.gen_soup(20000, 4)
    lights = np.array([light((1.0, 0.9, 0.8), (0.3, -1.0, 0.2), 1.5)], np.float32) if look == "lights" else None
    own.upload_scene(tris, infos, settings=ptamd.Settings(5, 2, 1.0, 1), lights=lights)
    if look == "detail":
        own.upload_detail(*random_detail(len(infos), 5))
    before = beside()
    want = play(own, sizes, sync=True)
    assert beside() == before
    for _ in range(2):
        before = beside()
        got = play(own, sizes, sync=False)
        assert beside() - before > SLOTS
        np.testing.assert_array_equal(got[0], want[0])
        assert got[1:] == want[1:] and np.any(want[0] != 0)
    assert own.get_status() == 0


def test_screen_buffer_and_streams(own):
    """The image written after every frame, on the context's stream and on a
    caller's, and after going back."""
    tris, infos = ptamd.gen_soup(20000, 4)
    own.upload_scene(tris, infos, settings=ptamd.Settings(5, 2, 1.0, 1))
    w, h = 160, 120
    screen = hip.DeviceArray((h, w, 4), np.float32)
    own.set_screen_buffer(screen.ptr, w, h)
    stream = hip.Stream()
    images = {}
    for sync in (True, False):
        images[sync] = []
        for s in (None, stream.handle, None):
            print(f"[beside] screen buffer, sync {sync}, stream {s}", flush=True)
            own.set_stream(s)
            before = beside()
            play(own, [(w, h)] * 8, sync)
            own.synchronize()
            assert sync or beside() - before > SLOTS
            images[sync].append(screen.to_host())
    own.set_stream(None)
    own.set_screen_buffer(0)
    stream.destroy()
    for a, b in zip(images[True], images[False]):
        np.testing.assert_array_equal(a, b)
    assert np.any(images[True][0] != 0)


def test_reported_time_is_the_frames(own):
    """A frame beside a long one reports no less than such a frame takes alone
    (within 30 %, for clocks), though little of it is left when the long one ends."""
    tris, infos = ptamd.gen_soup(65536, 4)
    own.upload_scene(tris, infos, settings=ptamd.Settings(6, ptamd.INVALID, 1.0, 1))
    w, h = 160, 120
    cam = camera(w, h, 0)
    own.set_primary_rays(cam, EYE)
    alone = []
    for k in range(6):
        own.synchronize()
        own.render_pass(w, h, k)
        alone.append(own.last_render_ms())
    many = np.stack([cam] * 200)
    own.synchronize()
    before = beside()
    own.render_passes(w, h, np.arange(200, dtype=np.uint64), many)
    own.render_pass(w, h, 7)
    ms = own.last_render_ms()
    print(f"[beside] alone {min(alone[1:]):.3f} ms, beside a long frame {ms:.3f} ms", flush=True)
    assert beside() == before + 1
    assert ms > 0.7 * min(alone[1:])
