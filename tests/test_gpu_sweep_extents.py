"""3D plans on fine grids off the sweep's 8-cell blocks, which are stored with
larger extents: the z-sweep spread and the z-gather there against the tile
kernels on the periodic grid, the fold and fill of the overhang at its edges
(points on the period's ends), batches, disjoint groups, re-pointing, and
crowded point sets, which go to the tiles."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _cplx(rng, shape):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)


def _pts(rng, M, edge=False):
    x = [rng.uniform(-np.pi, np.pi, M) for _ in range(3)]
    if edge:  # within a cell or two of the period's ends, and exactly on them
        for d, v in enumerate(x):
            s = slice(d * M // 8, (d + 1) * M // 8 + M // 64)
            n = v[s].size
            v[s] = rng.choice([-1, 1], n) * (np.pi - rng.uniform(0, 0.1, n))
            v[:3] = (np.pi, -np.pi, 0.0)
    return tuple(x)


# eps 1e-1 .. 1e-7: w = 2 .. 8
@pytest.mark.parametrize("N,eps,M,edge", [
    ((9, 11, 13), 1e-1, 3000, False), ((9, 25, 10), 1e-2, 3000, True),
    ((25, 9, 27), 1e-3, 5000, True), ((25, 15, 9), 1e-4, 1, False),
    ((27, 25, 33), 1e-5, 20000, False), ((10, 27, 45), 1e-6, 2000, True),
    ((45, 10, 9), 1e-6, 1500, True), ((27, 15, 25), 1e-7, 3000, True),
])
def test_extents_match_tiles(N, eps, M, edge, mn):
    print(f"case extents N={N} eps={eps} M={M} edge={edge}", flush=True)
    rng = np.random.default_rng(31)
    x, c, f = _pts(rng, M, edge), _cplx(rng, M), _cplx(rng, N)
    p = mn.Type1PlanND(x, N, eps=eps)
    q = mn.Type1PlanND(x, N, eps=eps, spread_method="gm")
    assert p.pts.kind == "zsweep" and p._store() is not None and q.pts.kind == "tiles"
    a, b = p.execute(c), q.execute(c)
    # fp32 weights, split products and sums against fp64 ones: a few 2^-24 of
    # exponent error (times beta <= 18.4) per axis and 2^-22 per product
    tol = 3 * 4 * 2.0 ** -24 * p.beta + 2.0 ** -21
    assert np.linalg.norm(a - b) <= tol * np.linalg.norm(b)
    cs = _cplx(rng, (3, M))
    s = p.execute_batch(cs)
    for k in range(3):
        one = p.execute(cs[k])
        assert np.linalg.norm(s[k] - one) <= 1e-6 * np.linalg.norm(one)
    # the adjoint over the same extents, where points are dense enough for it
    g = mn.Type2PlanND(x, N, eps=eps)
    h = mn.Type2PlanND(x, N, eps=eps, spread_method="gm")
    u, v = g.execute(f), h.execute(f)
    assert np.linalg.norm(u - v) <= tol * np.linalg.norm(v)


@pytest.mark.parametrize("N,eps,M", [((9, 11, 13), 1e-6, 3000), ((27, 25, 33), 1e-5, 60000),
                                     ((10, 27, 45), 1e-7, 10000)])
def test_extents_gather_and_oracle(N, eps, M, oracle, mn):
    print(f"case extents gather N={N} eps={eps} M={M}", flush=True)
    rng = np.random.default_rng(32)
    x, f, c = _pts(rng, M), _cplx(rng, N), _cplx(rng, M)
    g = mn.Type2PlanND(x, N, eps=eps)
    assert g.pts.kind == "zgather" and g._store() is not None
    idx = np.arange(0, M, 61)
    exact = oracle.dft_t2(x, f, -1, idx)
    ref = oracle.rel_l2(oracle.nufft_t2(x, f, eps, -1)[idx], exact)
    assert oracle.rel_l2(g.execute(f)[idx], exact) <= max(eps, 2 * ref)
    p = mn.Type1PlanND(x, N, eps=eps)
    ks = [np.arange(-(n // 2), n - n // 2) for n in N]
    e1 = oracle.dft_t1(x, c, ks, +1)
    ref1 = oracle.rel_l2(oracle.nufft_t1(x, c, N, eps, +1), e1)
    assert oracle.rel_l2(p.execute(c), e1) <= max(eps, 2 * ref1)


def test_extents_repoint_crowded_and_disjoint(mn):
    """A plan on extents follows its point sets: spread out (sweep), crowded
    (tiles), spread out again, each equal to a fresh plan; disjoint groups
    equal the groups' own transforms."""
    print("case extents repoint", flush=True)
    rng = np.random.default_rng(33)
    N, M, eps = (27, 25, 33), 40000, 1e-5
    p = mn.Type1PlanND(_pts(rng, M), N, eps=eps)
    crowd = tuple(rng.uniform(0.1, 0.2, M) for _ in range(3))
    for x, kind in ((crowd, "tiles"), (_pts(rng, M), "zsweep"), (_pts(rng, M // 3), "zsweep")):
        c = _cplx(rng, x[0].size)
        p.set_sources(x)
        assert p.pts.kind == kind
        ref = mn.Type1PlanND(x, N, eps=eps, spread_method="gm").execute(c)
        assert np.linalg.norm(p.execute(c) - ref) <= 3e-6 * np.linalg.norm(ref)
    groups = rng.choice([0, 1, -1], x[0].size)
    out = p.execute_disjoint(c, groups)
    for k in range(2):
        m = groups == k
        ref = mn.Type1PlanND(tuple(v[m] for v in x), N, eps=eps, spread_method="gm").execute(c[m])
        assert np.linalg.norm(out[k] - ref) <= 3e-6 * np.linalg.norm(ref)


def test_crowded_points_on_native_grids(mn):
    """From 2^18 points on, crowded sets leave the sweep and the z-gather on
    their own grids too, and come back when the points spread out."""
    print("case crowded native", flush=True)
    rng = np.random.default_rng(34)
    N, M, eps = (32, 32, 32), 1 << 18, 1e-6
    crowd = tuple(rng.uniform(0.1, 0.3, M) for _ in range(3))
    wide, c, f = _pts(rng, M), _cplx(rng, M), _cplx(rng, N)
    p = mn.Type1PlanND(crowd, N, eps=eps)
    g = mn.Type2PlanND(crowd, N, eps=eps)
    assert p.pts.kind == "tiles" and g.pts.kind == "tiles"
    ref = mn.Type1PlanND(crowd, N, eps=eps, spread_method="gm").execute(c)
    assert np.linalg.norm(p.execute(c) - ref) <= 3e-6 * np.linalg.norm(ref)
    ref = mn.Type2PlanND(crowd, N, eps=eps, spread_method="gm").execute(f)
    assert np.linalg.norm(g.execute(f) - ref) <= 3e-6 * np.linalg.norm(ref)
    p.set_sources(wide)
    assert p.pts.kind == "zsweep"
    ref = mn.Type1PlanND(wide, N, eps=eps, spread_method="gm").execute(c)
    assert np.linalg.norm(p.execute(c) - ref) <= 3e-6 * np.linalg.norm(ref)


def test_crowded_points_2d(mn):
    """The 2D sweep hands crowded sets of 2^17 points or more to the tiles, and
    grids that only the VALU y-sweep fits go to them when they are dense."""
    print("case crowded 2d", flush=True)
    rng = np.random.default_rng(35)
    M, eps = 1 << 17, 1e-6
    crowd = tuple(rng.uniform(0.1, 0.2, M) for _ in range(2))
    wide, c = tuple(rng.uniform(-np.pi, np.pi, M) for _ in range(2)), _cplx(rng, M)
    p = mn.Type1PlanND(crowd, (128, 128), eps=eps)
    for x, kind in ((crowd, "tiles"), (wide, "ymfma"), (wide, "ymfma")):
        p.set_sources(x)
        assert p.pts.kind == kind
        ref = mn.Type1PlanND(x, (128, 128), eps=eps, spread_method="gm").execute(c)
        assert np.linalg.norm(p.execute(c) - ref) <= 3e-6 * np.linalg.norm(ref)
    q = mn.Type1PlanND(wide, (128, 135), eps=eps)     # 256 x 270
    assert q.pts.kind == "tiles"
