"""How far CCD searches get, by the counters of the tiers, with the outcomes
against the oracle: sub-wave, wave, workgroup, lists past LDS and the
level-by-level wavefront.  Times of impact and steps are dyadic corners that
both sides compute exactly, so they must be equal."""
import numpy as np
import pytest

from test_gpu_parity import make, say, upload

pytestmark = pytest.mark.gpu

NAMES = ("spilled", "past_sub", "wavefront", "past_wide", "slabs", "by_level")


def reached(ctx):
    n = {k: ctx.counter("ccd." + k) for k in NAMES}
    say("reached", n)
    return {k for k in NAMES if n[k] > 0}


# bounded searches: tiers that every run reaches (how many searches get there
# depends on the order in which outcomes arrive)
@pytest.mark.parametrize("name,tiers", [
    ("twisted:8:0", {"wavefront"}),                             # a wave each at once
    ("stack:24:4", {"spilled", "wavefront"}),                   # no sub-wave tier
    ("sheets:48:2", {"spilled", "past_sub", "wavefront", "past_wide", "slabs"}),
    ("twisted:64:0", {"spilled", "past_sub", "wavefront", "past_wide", "slabs"}),
    ("sheets:10:0", {"spilled", "wavefront", "past_wide", "slabs", "by_level"}),
])
def test_step(ctx, O, scenes, name, tiers):
    s = make(scenes, name)
    say("case", name)
    upload(ctx, s)
    want = O.compute_collision_free_stepsize(s.V, s.V1, s.E, s.F)
    for _ in range(2):  # (the first call may reserve all lists past LDS)
        assert ctx.stepsize() == want
        assert reached(ctx) >= tiers
    assert ctx.is_step_collision_free() == (want == 1.0)


# searches without a bound: the counts do not depend on their order, except
# for who gets the lists past LDS
@pytest.mark.parametrize("name,limit,tiers", [
    ("stack:24:4", 20_000, {"spilled", "wavefront"}),
    ("twisted:16:0", 6000, {"spilled", "wavefront", "past_wide", "slabs"}),
    ("sheets:8:3", 20_000, {"spilled", "wavefront", "past_wide", "slabs", "by_level"}),
    ("sheets:16:0", 400, {"spilled", "past_sub", "wavefront", "past_wide", "slabs", "by_level"}),
])
def test_times_of_impact(ctx, O, scenes, name, limit, tiers):
    s = make(scenes, name)
    say("case", name, limit)
    upload(ctx, s)
    ctx.broad_phase(True, 0.0)
    ee, fv = ctx.candidates()
    p = O.CCDParams(1e-6, limit, 0.8)
    oe = O.candidates_toi(s.V, s.V1, s.E, s.F, ee, True, params=p)
    of = O.candidates_toi(s.V, s.V1, s.E, s.F, fv, False, params=p)
    for _ in range(2):
        te, tf = ctx.candidates_toi(max_iterations=limit)
        assert np.array_equal(te, oe) and np.array_equal(tf, of)
        assert reached(ctx) == tiers


def test_many_long_searches_advance_together(ctx, O, scenes):
    """more than 4096 searches left without a bound skip the workgroup tier"""
    s = make(scenes, "sheets:16:0")
    say("case many")
    upload(ctx, s)
    ctx.broad_phase(True, 0.0)
    ee, _ = ctx.candidates()
    te, _ = ctx.candidates_toi(max_iterations=6000)
    assert reached(ctx) == {"spilled", "past_sub", "wavefront", "past_wide", "by_level"}
    assert ctx.counter("ccd.by_level") > 4096
    p = O.CCDParams(1e-6, 6000, 0.8)
    assert np.array_equal(te, O.candidates_toi(s.V, s.V1, s.E, s.F, ee, True, params=p))


def test_lists_past_lds_are_reserved_when_asked_for(ctx, O, scenes):
    for name, few in (("stack:24:4", False), ("twisted:32:0", True)):
        s = make(scenes, name)
        say("case memory", name)
        upload(ctx, s)
        assert ctx.stepsize() == O.compute_collision_free_stepsize(s.V, s.V1, s.E, s.F)
        assert ("slabs" in reached(ctx)) == few
        small = ctx.device_bytes()
        say("device bytes", small)
        assert small < 32 << 20  # all lists are 42 MB
    s = make(scenes, "sheets:10:0")
    upload(ctx, s)
    assert ctx.stepsize() == O.compute_collision_free_stepsize(s.V, s.V1, s.E, s.F)
    assert "slabs" in reached(ctx) and ctx.device_bytes() > small + (32 << 20)


def test_more_searches_than_the_box_budget_is_for(ctx, capi, scenes):
    """past 2^25 searches a lane's search is not cut at 24 boxes; the steps are
    those of each scene alone"""
    B = scenes.Batch(scenes.batch_scenes(48, seed=0))
    say("batch", len(B.scenes), B.sizes)
    ctx.upload_batch(B)
    ctx.upload_positions(0, B.V)
    ctx.upload_positions(1, B.V1)
    steps = ctx.stepsize_batched()
    assert ctx.counter("ccd.searched") > 1 << 25
    alone = capi.Context(0)
    try:
        for k in np.argsort([len(s.F) for s in B.scenes])[::5]:
            upload(alone, B.scenes[k])
            assert alone.stepsize() == steps[k], k
            assert alone.counter("ccd.searched") < 1 << 25
    finally:
        alone.close()
