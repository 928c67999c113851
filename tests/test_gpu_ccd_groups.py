"""CCD searches that outgrow a lane's lists: the sub-wave, wave, workgroup
and wavefront tiers against the oracle.  Times of impact and steps are
dyadic corners that both sides compute exactly, so they must be equal."""
import numpy as np
import pytest

from test_gpu_parity import make, say, upload

pytestmark = pytest.mark.gpu


# searches: under 4096 (a wave each at once), spilled lists under and over the
# sub-wave tier's threshold, levels past a workgroup's LDS lists
STEPS = ["twisted:8:0", "sheets:8:3", "sheets:20:1", "sheets:48:2", "spheres:5:3:7", "stack:24:4"]


@pytest.mark.parametrize("name", STEPS)
def test_step(ctx, O, scenes, name):
    s = make(scenes, name)
    say("case", name, s.sizes)
    upload(ctx, s)
    for md in (0.0, 1e-5):
        t = ctx.stepsize(min_distance=md)
        assert t == O.compute_collision_free_stepsize(s.V, s.V1, s.E, s.F, min_distance=md)
        assert ctx.counter("ccd.unmet") == 0
        assert ctx.is_step_collision_free(min_distance=md) == (t == 1.0)
    # a step that stays free of collisions, and one twice as long
    for f in (0.05, 2.0):
        V1 = s.V + f * (s.V1 - s.V)
        ctx.upload_positions(1, V1)
        t = ctx.stepsize()
        assert t == O.compute_collision_free_stepsize(s.V, V1, s.E, s.F)
        assert ctx.is_step_collision_free() == (t == 1.0)


@pytest.mark.parametrize("max_iter", [1, 2, 37, 400, 20_000])
@pytest.mark.parametrize("name", ["tet", "twisted:8:0", "sheets:8:3", "spheres:4:3:0"])
def test_iteration_limit(ctx, O, scenes, name, max_iter):
    """per-candidate times (no bound between candidates) where the limit
    ends searches inside every tier"""
    s = make(scenes, name)
    say("case", name, max_iter)
    upload(ctx, s)
    ctx.broad_phase(True, 0.0)
    ee, fv = ctx.candidates()
    te, tf = ctx.candidates_toi(max_iterations=max_iter)
    p = O.CCDParams(1e-6, max_iter, 0.8)
    assert np.array_equal(te, O.candidates_toi(s.V, s.V1, s.E, s.F, ee, True, params=p))
    assert np.array_equal(tf, O.candidates_toi(s.V, s.V1, s.E, s.F, fv, False, params=p))


@pytest.mark.parametrize("gap", [1e-9, 1e-7, 3e-6])
@pytest.mark.parametrize("n", [8, 40])
def test_restart_near_contact(ctx, O, scenes, n, gap):
    """sheets so close that first searches end below 1e-6 and start again
    from the minimum distance"""
    s = scenes.two_sheets(n, seed=n, twist=0.2)
    nb = len(s.V) // 2
    V, V1 = s.V.copy(), s.V1.copy()
    V[nb:, 2] = gap * (1.0 + np.arange(nb) % 3)
    V1[nb:] = V[nb:] + [2e-4, 1e-4, -1e-3]
    s = scenes.Scene("close", V, s.E, s.F, V1, s.dhat, s.kappa)
    say("case", n, gap)
    upload(ctx, s)
    t = ctx.stepsize()
    assert t == O.compute_collision_free_stepsize(V, V1, s.E, s.F)
    assert ctx.is_step_collision_free() == (t == 1.0)
