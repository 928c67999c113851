"""Broad phase and merge at the sizes where their launches change: arrays at
the edges of one workgroup's sort (8192 keys), of the sort's tiles, of the
refit's leaf ranges (1024 leaves, 64 of them) and a forest of uneven scenes.
Sets and orientations must equal the oracle's, on every call."""
import numpy as np
import pytest

from conftest import pair_set, sparse_rel_err
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


def soup(n, seed=0):
    """n small disjoint triangles (3 n vertices, 3 n edges, n faces) in a slab"""
    rng = np.random.default_rng([n, seed])
    side = np.sqrt(n) * 0.02
    c = rng.uniform(0, 1, (n, 1, 3)) * [side, side, 0.02]
    V = (c + rng.uniform(-0.01, 0.01, (n, 3, 3))).reshape(-1, 3)
    F = np.arange(3 * n, dtype=np.int32).reshape(-1, 3)
    E = np.stack([F[:, [0, 1]], F[:, [1, 2]], F[:, [0, 2]]], 1).reshape(-1, 2)
    return V, np.ascontiguousarray(E, np.int32), F


@pytest.mark.parametrize("n", [1, 2, 341, 342, 683, 1023, 1024, 1025, 2730, 2731, 8193, 21845,
                               21846, 43691])
def test_sets(ctx, O, n):
    V, E, F = soup(n)
    say("case", n)
    ctx.upload_mesh(V, E, F)
    ctx.upload_positions(0, V)
    dhat = 1.5e-3
    ctx.broad_phase(False, 0.5 * dhat)
    ee, fv = ctx.candidates()
    eo, fo = O.candidates(V, E, F, 0.5 * dhat)
    assert len(ee) == len(eo) and pair_set(ee) == pair_set(eo)
    assert len(fv) == len(fo) and pair_set(fv) == pair_set(fo)
    ctx.build_collisions(dhat)
    got, want = ctx.collisions(), O.build_collisions(V, E, F, eo, fo, dhat)
    for k in ("vv", "ev", "ee", "fv"):
        assert np.array_equal(got[k], getattr(want, k)), k
        assert np.array_equal(got[k + "_w"], getattr(want, k + "_w")), k
    # a repeated call and the sweep reuse the same scratch
    ctx.broad_phase(False, 0.5 * dhat, 0)
    again = ctx.candidates()
    for a, b in ((again[0], ee), (again[1], fv)):
        assert len(a) == len(b) and pair_set(a) == pair_set(b)
    ctx.broad_phase(False, 0.5 * dhat, 1)
    swept = ctx.candidates()
    for a, b in zip(swept, O.candidates(V, E, F, 0.5 * dhat, method="sap")):
        assert len(a) == len(b) and pair_set(a) == pair_set(b)


# one context through arrays of every sort path, up and down in size: 64-bit
# keys (trees, merges), 32-bit keys (incidences), scans and run lengths share
# look-back words, ticket and histograms with the calls before
@pytest.mark.parametrize("order", [[8193, 2, 21846, 1, 43691, 683, 8193],
                                   [43691, 43691, 5, 2731, 341, 21845, 1024],
                                   [1, 8193, 8193, 1, 8193, 2, 43691]])
def test_scratch_across_calls(ctx, O, order):
    for n in order:
        V, E, F = soup(n)
        say("case", order, n)
        ctx.upload_mesh(V, E, F)
        ctx.upload_positions(0, V)
        dhat = 1.5e-3
        eo, fo = O.candidates(V, E, F, 0.5 * dhat)
        want = O.build_collisions(V, E, F, eo, fo, dhat)
        Ho = O.barrier_hessian(want, V, E, F, dhat, 1e3, "clamp")
        for _ in range(2):
            ctx.build_collisions(dhat)
            ee, fv = ctx.candidates()
            assert len(ee) == len(eo) and pair_set(ee) == pair_set(eo)
            assert len(fv) == len(fo) and pair_set(fv) == pair_set(fo)
            got = ctx.collisions()
            for k in ("vv", "ev", "ee", "fv"):
                assert np.array_equal(got[k], getattr(want, k)), k
                assert np.array_equal(got[k + "_w"], getattr(want, k + "_w")), k
            assert sparse_rel_err(ctx.hessian(dhat, 1e3, "clamp"), Ho) <= 1e-10


@pytest.mark.parametrize("sizes", [(1, 1, 1), (1, 400, 2), (342, 1, 5000, 1, 341), (22000, 3, 700)])
def test_forest(ctx, capi, scenes, O, sizes):
    parts = [scenes.Scene(f"soup{n}", *soup(n, seed=k), soup(n, seed=k)[0], 1.5e-3, 1e3)
             for k, n in enumerate(sizes)]
    b = scenes.Batch(parts)
    say("case", sizes)
    ctx.upload_batch(b)
    ctx.upload_positions(0, b.V)
    ctx.broad_phase(False, 0.75e-3)
    ee, fv = ctx.candidates()
    eo, fo = [], []
    for k, s in enumerate(parts):
        e, f = O.candidates(s.V, s.E, s.F, 0.75e-3)
        eo.append(np.asarray(e).reshape(-1, 2) + b.eoff[k])
        fo.append(np.asarray(f).reshape(-1, 2) + [b.foff[k], b.voff[k]])
    assert pair_set(ee) == pair_set(np.concatenate(eo))
    assert pair_set(fv) == pair_set(np.concatenate(fo))
