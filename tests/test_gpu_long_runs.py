"""Real-valued merges with short and long runs of contributions to one pair,
and sub-element keys that fill a workgroup's buffer: two fans of triangles
apex to apex (about degree^2 contributions to the apex pair), against the oracle.  Both sides
sum in ascending order of value, so ids and weights are identical."""
import numpy as np
import pytest

from test_gpu_improved import assert_same_set, oracle_set

pytestmark = pytest.mark.gpu

DHAT = 1e-2


def fans(deg):
    rng = np.random.default_rng(deg)
    V, F = [], []
    for z in (1.0, -1.0):
        o = len(V)
        V.append([0, 0, z * 0.25 * DHAT])
        for k in range(deg):
            a = 2 * np.pi * k / deg
            V.append([np.cos(a) * rng.uniform(0.8, 1.2), np.sin(a) * rng.uniform(0.8, 1.2), z])
        F += [[o, o + 1 + k, o + 1 + (k + 1) % deg] for k in range(deg)]
    V, F = np.array(V), np.array(F, dtype=np.int32)
    E = np.unique(np.sort(np.concatenate([F[:, [0, 1]], F[:, [1, 2]], F[:, [2, 0]]]), axis=1),
                  axis=0).astype(np.int32)
    return V, E, F


# runs of up to 16, of a wave (up to 128) and longer
@pytest.mark.parametrize("deg", [3, 4, 5, 12, 22, 24, 40])
@pytest.mark.parametrize("improved", [False, True])
def test_runs_of_every_length(ctx, capi, O, deg, improved):
    V, E, F = fans(deg)
    ctx.upload_mesh(V, E, F)
    ctx.upload_positions(0, V)
    ctx.set_area_weighting(True)
    if improved:
        ctx.set_collision_set_type(capi.COLLISIONS_IMPROVED_MAX_APPROX)
    ctx.build_collisions(DHAT)
    co = oracle_set(ctx, O, V, E, F, DHAT, aw=True, improved=improved)
    print("case", deg, improved, [len(co.vv), len(co.ev), len(co.ee), len(co.fv)], flush=True)
    assert len(co.vv) == 1
    assert_same_set(ctx.collisions(), co)


@pytest.mark.parametrize("deg", [11, 12, 24])
def test_many_long_runs(ctx, capi, O, deg):
    """300 apex pairs of a run each at both sides of a wave's buffer, all of
    them in a few waves: equal weights, and not one long run after the other (24
    triangles an apex took 2.8 s then)"""
    V0, E0, F0 = fans(deg)
    n = 300
    V = np.concatenate([V0 + [4.0 * (k % 20), 4.0 * (k // 20), 0] for k in range(n)])
    E = np.concatenate([E0 + len(V0) * k for k in range(n)]).astype(np.int32)
    F = np.concatenate([F0 + len(V0) * k for k in range(n)]).astype(np.int32)
    ctx.upload_mesh(V, E, F)
    ctx.upload_positions(0, V)
    ctx.set_area_weighting(True)
    ctx.build_collisions(DHAT)
    ctx.timing(True)
    ctx.build_collisions(DHAT)
    ms = ctx.stage_times()["np_merge"][0]
    ctx.timing(False)
    got = ctx.collisions()
    print("case many", ms, [len(got[k]) for k in ("vv", "ev", "ee", "fv")], flush=True)
    assert_same_set(got, oracle_set(ctx, O, V, E, F, DHAT, aw=True, improved=False))
    assert len(got["vv"]) == n and ms < 100
