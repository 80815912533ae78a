"""The autotuner's staged search: stages of knobs that a frame structure does not
read are left out, the others are searched in order.  (Times are made up: no
GPU.)
"""
import pytest

import ptamd
from ptamd import autotune

KNOBS = ("render.paths", "render.chains", "render.shade_min", "render.shade_lit", "render.refill", "trace.blocks",
         "trace.lds_stack", "trace.refill", "trace.pool")


@pytest.fixture
def saved():
    before = {k: ptamd.tune_get(k) for k in KNOBS}
    yield
    for k, v in before.items():
        ptamd.tune_set(k, v)


@pytest.mark.parametrize("paths", [0, 1])
def test_queue_knobs_only_for_bounce_levels(saved, monkeypatch, paths):
    # Faster at the structure wanted, at fewer blocks, and at the first pool and refill.
    monkeypatch.setattr(autotune, "_time", lambda run, stream, reps: (
        (0.0 if ptamd.tune_get("render.paths") == paths else 100.0) + ptamd.tune_get("trace.blocks") / 1000.0
        + ptamd.tune_get("trace.pool") / 1000.0 + ptamd.tune_get("trace.refill") / 100.0))
    ptamd.tune_set("trace.pool", 512)
    stages = autotune.render_stages(64)
    assert {k for st in stages for k in st} == set(KNOBS)
    best, table = autotune.tune_staged(lambda: None, 0, stages)
    searched = {k for setting, _ in table for k in setting}
    assert best["render.paths"] == paths and best["trace.blocks"] == 64 * 6
    assert ("trace.pool" in searched) == ("trace.refill" in searched) == (paths == 0)
    assert ptamd.tune_get("trace.pool") == (128 if paths == 0 else 512)
    assert ptamd.tune_get("render.paths") == paths
