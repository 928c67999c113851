"""Hessian records by the frame of the closest points, and the rows that
expand them, against the CPU oracle: every stencil kind and edge-edge type,
with and without a mollifier, one collision and rows of several column
windows.  The bound is the contract's 1e-10 of the Frobenius norm (triangles
are kept fat: both sides lose |u| |v| / |u x v| roundings, the oracle's
point-space derivatives as much as the frame)."""
import numpy as np
import pytest

from conftest import sparse_rel_err

pytestmark = pytest.mark.gpu

DHAT, KAPPA = 2e-2, 1e3


def unit(rng):
    v = rng.normal(size=3)
    return v / np.linalg.norm(v)


def triangle(rng):
    a = unit(rng)
    b = np.cross(a, unit(rng))
    b /= np.linalg.norm(b)
    return 0.1 * np.array([[0, 0, 0], a, 0.4 * a + rng.uniform(0.6, 1.0) * b])


def soup(rng, groups, flat):
    """Pairs of triangles 10 apart, touching zone inside DHAT; flat: the
    second one parallel to the first (mollified edge pairs)."""
    P = []
    for g in range(groups):
        A = triangle(rng)
        n = np.cross(A[1], A[2])
        n /= np.linalg.norm(n)
        B = A @ np.diag([1, 1, 1]) if flat else triangle(rng)
        B = B - B[rng.integers(0, 3)] * rng.uniform(0, 1)
        w = rng.dirichlet([0.6, 0.6, 0.6])
        d = n if flat else unit(rng)
        at = np.array([10.0 * g, 0, 0])
        P += [A + at, B + w @ A + d * DHAT * rng.uniform(0.2, 0.9) + at]
    V = np.concatenate(P)
    return V, np.arange(len(V), dtype=np.int32).reshape(-1, 3)


def fan(rng, n):
    """n triangles through a small region: rows of more than 64 columns"""
    V = np.concatenate([triangle(rng) - 0.05 + 0.004 * rng.normal(size=3) for _ in range(n)])
    return V, np.arange(len(V), dtype=np.int32).reshape(-1, 3)


# (with a minimum separation only where no pair is closer: the barrier is
# infinite there)
@pytest.mark.parametrize("shape,dmin", [("one", 0.0), ("one", 1e-3), ("soup", 0.0), ("flat", 0.0),
                                        ("flat", 1e-3), ("fan", 0.0)])
def test_hessian_of_every_stencil(ctx, O, shape, dmin):
    rng = np.random.default_rng(11)
    V, F = {"one": lambda: (np.array([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0.2, 0.3, 5e-3],
                                      [0.3, 0.2, 2.0], [0.1, 0.2, 2.0]]),
                            np.arange(6, dtype=np.int32).reshape(-1, 3)),
            "soup": lambda: soup(rng, 400, False), "flat": lambda: soup(rng, 100, True),
            "fan": lambda: fan(rng, 40)}[shape]()
    E = np.unique(np.sort(np.concatenate([F[:, [0, 1]], F[:, [1, 2]], F[:, [2, 0]]]), axis=1),
                  axis=0).astype(np.int32)
    ctx.upload_mesh(V, E, F)
    ctx.upload_positions(0, V)
    ctx.upload_positions(1, V)
    ctx.build_collisions(DHAT, dmin)
    ee, fv = O.candidates(V, E, F, 0.5 * (DHAT + dmin))
    co = O.build_collisions(V, E, F, ee, fv, DHAT, dmin)
    counts = [int(x) for x in ctx.collision_counts()]
    print("case", shape, dmin, counts, flush=True)
    if shape == "one":
        assert sum(counts) == 1
    else:
        assert min(counts) > 0
    for psd in ("none", "clamp", "abs"):
        Ho = O.barrier_hessian(co, V, E, F, DHAT, KAPPA, psd)
        Hg = ctx.hessian(DHAT, KAPPA, psd)
        assert sparse_rel_err(Hg, Ho) <= 1e-10, psd
        if shape == "fan":
            assert np.diff(Hg.indptr).max() > 3 * 64
    if shape == "flat":
        assert ctx.counter("hessian.ee_other") > 0
    if shape == "soup":
        assert ctx.counter("hessian.ee_other") < counts[2]  # mostly the closed form


ALONE = {  # one collision of one kind: the launch over the kinds has a single workgroup
    "vv": ([[0, 0, 0], [0, 0, 1], [0, 1, 0.5], [-5e-3, 0, 0], [-1, 0, 0.2], [-1, 1, 0.2]],
           [[0, 1, 2], [3, 4, 5]]),
    "fv": ([[0, 0, 0], [1, 0, 0], [0, 1, 0], [0.2, 0.3, 5e-3], [0.3, 0.2, 2.0], [0.1, 0.2, 2.0]],
           [[0, 1, 2], [3, 4, 5]]),
    "ee": ([[0, 0, 0], [1, 0, 0], [0.5, 0, -1], [0.4, -0.5, 5e-3], [0.5, 0.6, 5e-3], [0.5, 0, 1]],
           [[0, 1, 2], [3, 4, 5]]),
}


@pytest.mark.parametrize("kind", sorted(ALONE))
def test_one_kind_alone(ctx, O, kind):
    V, F = np.array(ALONE[kind][0], float), np.array(ALONE[kind][1], np.int32)
    E = np.unique(np.sort(np.concatenate([F[:, [0, 1]], F[:, [1, 2]], F[:, [2, 0]]]), axis=1),
                  axis=0).astype(np.int32)
    ctx.upload_mesh(V, E, F)
    ctx.upload_positions(0, V)
    ctx.build_collisions(DHAT)
    ee, fv = O.candidates(V, E, F, 0.5 * DHAT)
    co = O.build_collisions(V, E, F, ee, fv, DHAT)
    counts = dict(zip(("vv", "ev", "ee", "fv"), (int(x) for x in ctx.collision_counts())))
    print("case", kind, counts, flush=True)
    assert counts == {k: int(k == kind) for k in counts}
    e = O.barrier_energy(co, V, E, F, DHAT, KAPPA)
    assert abs(ctx.energy(DHAT, KAPPA) - e) <= 1e-12 * abs(e)
    g = O.barrier_gradient(co, V, E, F, DHAT, KAPPA)
    assert np.linalg.norm(ctx.gradient(DHAT, KAPPA).ravel() - g.ravel()) <= 1e-12 * np.linalg.norm(g)
    assert sparse_rel_err(ctx.hessian(DHAT, KAPPA, "clamp"),
                          O.barrier_hessian(co, V, E, F, DHAT, KAPPA, "clamp")) <= 1e-10
