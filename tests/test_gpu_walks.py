"""Tree walks: waves that start with 8, 16 or 64 queries, subtrees handed
between lanes, the queue of overlapping leaves and edge-edge beside
face-vertex walks in one launch, against the oracle's candidates and the
launches of the autotuned path.  Candidate sets are exact."""
import numpy as np
import pytest

from conftest import pair_set

pytestmark = pytest.mark.gpu


def pile(n):
    """n triangles through one another: every wave's queue fills at each
    step, and all the work belongs to few lanes"""
    rng = np.random.default_rng(5)
    V = rng.normal(size=(3 * n, 3))
    F = np.arange(3 * n, dtype=np.int32).reshape(-1, 3)
    return V, F


def edges(F):
    return np.unique(np.sort(np.concatenate([F[:, [0, 1]], F[:, [1, 2]], F[:, [2, 0]]]), axis=1),
                     axis=0).astype(np.int32)


def check(ctx, O, V, E, F, r):
    ctx.upload_mesh(V, E, F)
    ctx.upload_positions(0, V)
    ctx.broad_phase(False, r)
    ee, fv = ctx.candidates()
    ee_o, fv_o = O.candidates(V, E, F, r)
    assert len(ee) == len(ee_o) and pair_set(ee) == pair_set(ee_o)
    assert len(fv) == len(fv_o) and pair_set(fv) == pair_set(fv_o)
    return ee, fv


@pytest.mark.parametrize("n", [2, 5, 22, 64, 150])
def test_pile_of_triangles(ctx, O, n):
    V, F = pile(n)
    check(ctx, O, V, edges(F), F, 1e-3)


# nE + nV just below and above 2^16 and 2^18 (a sheet of n^2 vertices has
# 4 n^2 - 4 n + 1 of them)
@pytest.mark.parametrize("n", [128, 129, 256, 257])
def test_walks_at_the_limits_of_the_starting_widths(ctx, O, scenes, n):
    s = scenes.stacked_sheets(n, 1, seed=2, h=1.0 / 511)
    V = s.V.copy()
    V[::7] *= 0.98  # some far overlaps
    print("case", n, len(s.E) + len(V), flush=True)
    ee, fv = check(ctx, O, V, s.E, s.F, 0.5 * s.dhat)
    ctx.set_autotune(True)
    try:
        ctx.broad_phase(False, 0.5 * s.dhat)
        ee2, fv2 = ctx.candidates()
    finally:
        ctx.set_autotune(False)
    assert pair_set(ee) == pair_set(ee2) and pair_set(fv) == pair_set(fv2)


def comb(spokes):
    """Spokes from a corner hub, each spanning half the box, beside edges in
    20 octaves towards the spokes' centres: a walk from a spoke postpones the
    upper octave at each of 18 levels, more than a lane holds in LDS."""
    rng = np.random.default_rng(spokes)
    rim = 0.5 - 1e-6 * rng.uniform(0.1, 1, (spokes, 3))
    c = (0.25 + 0.25 * 2.0 ** -np.arange(20)[:, None] * [1.0, 1.3]).ravel()
    ends = c[:, None, None] + np.array([[-1e-9] * 3, [1e-9] * 3])
    V = np.concatenate([[[0, 0, 0]], rim, ends.reshape(-1, 3), [[1, 1, 0.999], [1, 1, 1]]])
    pairs = np.arange(spokes + 1, len(V)).reshape(-1, 2)
    E = np.concatenate([np.stack([np.zeros(spokes), np.arange(1, spokes + 1)], 1), pairs])
    return V, E.astype(np.int32), np.zeros((0, 3), np.int32)


# spill stacks claimed from the first pool, and more of them than it has
@pytest.mark.parametrize("spokes,least", [(40, 1), (12000, 1025)])
def test_spill_stacks(ctx, O, spokes, least):
    V, E, F = comb(spokes)
    print("case", spokes, flush=True)
    for _ in range(2):  # the second walk finds the pool at its size
        ee, fv = check(ctx, O, V, E, F, 1e-12)
        assert len(ee) >= 18 * 2 * spokes and len(fv) == 0
        assert ctx.counter("bp.spill_stacks") >= least


def test_tuned_walks_share_a_launch(ctx, scenes):
    """the tuner chooses the workgroup size of the launch that holds both
    walks; the names of the walks answer for it"""
    s = scenes.two_sheets(40, seed=3)
    ctx.upload_mesh(s.V, s.E, s.F)
    ctx.upload_positions(0, s.V)
    ctx.set_autotune(True)
    for _ in range(2):
        ctx.timing(True)
        ctx.broad_phase(False, 0.5 * s.dhat)
        names = set(ctx.stage_times())
        ctx.timing(False)
        print("stages", sorted(names), flush=True)
        assert "bp_traverse_both.static" in names and "bp_traverse_ee.static" not in names
    b, ms = ctx.launch_shape("bp_traverse_both.static")
    assert b in (64, 128, 256) and ms > 0
    assert ctx.launch_shape("bp_traverse_ee.static") == (b, ms)
    assert ctx.launch_shape("bp_traverse_fv.static") == (b, ms)
    assert ctx.launch_shape("bp_traverse_both.swept")[0] == 0
    # a mesh without faces: the edge-edge walk by itself
    ctx.upload_mesh(s.V, s.E, s.F[:0])
    ctx.upload_positions(0, s.V)
    ctx.broad_phase(False, 0.5 * s.dhat)
    assert ctx.launch_shape("bp_traverse_ee.static")[0] in (64, 128, 256)
