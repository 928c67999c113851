"""Expected minimums: where they do not stand, and the iteration limits that
search without one.  Two edges in near contact, their
coordinates large against the gap: the first search ends at time 0 (the
rounding filter fills the gap) and starts again from the minimum distance.
CUT: the search outgrows a wave's lists on the way, so its earliest boxes
alone give its scene an expected minimum (0.625, 0.0625, 0.0078) that the
second search does not meet (no hit, 0.1, 0.025).  KEPT: the search fits a wave's
lists, so its restart says nothing about the scenes' expected minimums."""
import numpy as np
import pytest

from test_gpu_parity import make, say, upload

pytestmark = pytest.mark.gpu

# edge a, edge b at the start, then at the end of the step
CUT = {
    "free": (
        [[10.918196152620146, 10.918196152620146, 10.918196152620146],
         [10.918196152961197, 10.918196151487511, 10.918196153100073],
         [10.918196152667145, 10.918196152535803, 10.918196152679522],
         [10.918196153024148, 10.918196151414897, 10.918196153175799]],
        [[10.918196152620146, 10.918196152620146, 10.918196152620146],
         [10.918196152961197, 10.918196151487511, 10.918196153100073],
         [10.918196152664969, 10.918196152517035, 10.91819615267891],
         [10.918196153006935, 10.91819615138507, 10.918196153159775]],
    ),
    "tenth": (
        [[44.930573839341065, 44.930573839341065, 44.930573839341065],
         [44.930573911249006, 44.93057370750094, 44.930573886092773],
         [44.930573851169868, 44.930573820965996, 44.930573847440677],
         [44.930573923861303, 44.930573689827455, 44.930573894965768]],
        [[44.930573839341065, 44.930573839341065, 44.930573839341065],
         [44.930573911249006, 44.93057370750094, 44.930573886092773],
         [44.930573847828832, 44.930573816856729, 44.93057384400479],
         [44.930573926600431, 44.930573691162664, 44.930573897531559]],
    ),
    "fortieth": (
        [[27.51294998330059, 27.51294998330059, 27.51294998330059],
         [27.512950022023361, 27.512949956065512, 27.512949984627049],
         [27.512949977422771, 27.512949987893059, 27.512949983359139],
         [27.512950016138984, 27.512949960648257, 27.512949984677245]],
        [[27.51294998330059, 27.51294998330059, 27.51294998330059],
         [27.512950022023361, 27.512949956065512, 27.512949984627049],
         [27.51294997208532, 27.512949980324432, 27.512949976756673],
         [27.51295002295819, 27.512949971118445, 27.512949993566462]],
    ),
}
KEPT = {
    "pair": (
        [[42.946228067583505, 42.946228067583505, 42.946228067583505],
         [42.946228073005244, 42.946228062291574, 42.946228066154795],
         [42.946228069513609, 42.946228067278483, 42.946228068084444],
         [42.946228076116611, 42.946228062920568, 42.946228067678895]],
        [[42.946228067583505, 42.946228067583505, 42.946228067583505],
         [42.946228073005244, 42.946228062291574, 42.946228066154795],
         [42.946228067383593, 42.946228066783085, 42.946228066999623],
         [42.946228078586017, 42.946228066061863, 42.946228070577916]],
    ),
}


def pair(scenes, which):
    V, V1 = (np.array(x) for x in which)
    return scenes.Scene("pair", V, [[0, 1], [2, 3]], np.zeros((0, 3), np.int32), V1, 1e-3, 1e3)


def oracle_steps(O, parts):
    return np.array([O.compute_collision_free_stepsize(s.V, s.V1, s.E, s.F) for s in parts])


@pytest.mark.parametrize("name", sorted(CUT))
def test_searched_again_without_it(ctx, O, scenes, name):
    s = pair(scenes, CUT[name])
    say("case", name)
    upload(ctx, s)
    t = ctx.stepsize()
    assert t == oracle_steps(O, [s])[0]
    assert ctx.counter("ccd.unmet") == 1
    assert ctx.is_step_collision_free() == (t == 1.0)


def test_restart_of_another_search(ctx, O, scenes):
    s = pair(scenes, KEPT["pair"])
    say("case kept")
    upload(ctx, s)
    assert ctx.stepsize() == oracle_steps(O, [s])[0]
    assert ctx.counter("ccd.unmet") == 0


def batched(ctx, O, scenes, parts):
    b = scenes.Batch(parts)
    say("batch", b.sizes)
    ctx.upload_batch(b)
    ctx.upload_positions(0, b.V)
    ctx.upload_positions(1, b.V1)
    assert np.array_equal(ctx.stepsize_batched(), oracle_steps(O, parts))
    return ctx.counter("ccd.unmet")


def test_restart_of_another_scene(ctx, O, scenes):
    """the sheets' expected minimums stand whatever the pair's search does"""
    parts = [make(scenes, "sheets:8:3"), pair(scenes, KEPT["pair"]), make(scenes, "sheets:12:1")]
    assert batched(ctx, O, scenes, parts) == 0


@pytest.mark.parametrize("big", [False, True])  # (big: past the direct wave tier)
def test_only_its_scenes_are_searched_again(ctx, O, scenes, big):
    parts = [make(scenes, "sheets:8:3"), pair(scenes, CUT["tenth"]), make(scenes, "twisted:8:0"),
             pair(scenes, CUT["free"])] + [make(scenes, "sheets:40:1")] * big
    assert batched(ctx, O, scenes, parts) == 2


@pytest.mark.parametrize("limit", [20_000, 999_999, 1_000_000, 9_999_999, 10_000_000, -1])
@pytest.mark.parametrize("seed", [0, 1])
def test_step_at_iteration_limits(ctx, O, scenes, seed, limit):
    """A minimum is expected from the default limit on.  A bound can only keep
    searches from meeting the limit, so the step lies between the smallest
    outcome of the searches alone and the step without a limit."""
    s = scenes.two_sheets(10, seed=seed)
    say("case limit", seed, limit)
    upload(ctx, s)
    t = ctx.stepsize(max_iterations=limit)
    assert ctx.counter("ccd.expected") == int(limit < 0 or limit >= 10_000_000)
    alone, free = (O.compute_collision_free_stepsize(s.V, s.V1, s.E, s.F,
                                                     params=O.CCDParams(1e-6, n, 0.8))
                   for n in (limit if limit > 0 else 10_000_000, 10_000_000))
    assert alone <= t <= free
    if limit < 0 or limit >= 10_000_000:
        assert t == free
