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


def _sums64(x, c, f, N, ntrg):
    """Direct type-1 sums, and type-2 sums at the first ntrg points, in 64 bits."""
    step = 8192
    t1 = torch.zeros(N[0] * N[1], N[2], dtype=torch.complex128, device="cuda")
    t2 = []
    fd = torch.from_numpy(f).cuda().to(torch.complex128).reshape(N[0], -1)
    for lo in range(0, x[0].size, step):
        e = []
        for d in range(3):
            k = torch.arange(-(N[d] // 2), N[d] - N[d] // 2, dtype=torch.float64, device="cuda")
            ph = torch.from_numpy(x[d][lo:lo + step]).cuda()[:, None] * k
            e.append(torch.complex(torch.cos(ph), torch.sin(ph)))
        cd = torch.from_numpy(c[lo:lo + step]).cuda().to(torch.complex128)
        xy = (e[0][:, :, None] * (cd[:, None] * e[1])[:, None, :]).reshape(cd.numel(), -1)
        t1 += xy.T.contiguous() @ e[2]
        if lo < ntrg:
            g = (e[0].conj().contiguous() @ fd).reshape(-1, N[1], N[2])
            t2.append(((g * e[1].conj()[:, :, None]).sum(1) * e[2].conj()).sum(1))
    return t1.reshape(N), torch.cat(t2)[:ntrg]


# eps, points per cell, most allowed relative error: what fp64 tile sums of
# fp32 weights gave here (1.45e-6 at w = 7, 6.9e-7 to 7.3e-7 at w = 8)
@pytest.mark.parametrize("eps,dens,most", [(1e-6, 0.3, 1.46e-6), (1e-6, 6.0, 1.46e-6),
                                           (1e-7, 0.3, 7.3e-7), (1e-7, 6.0, 7.3e-7)])
def test_extents_no_less_precise_than_fp64_sums(eps, dens, most, mn):
    """Split products and fp32 sums on extents against 64 bits, with strengths
    and modes of one size and over a range of e^+-12: no further off than fp64
    sums of fp32 weights on the periodic grid."""
    print(f"case extents precision eps={eps} points per cell {dens}", flush=True)
    rng = np.random.default_rng(36)
    N = (45, 50, 55)                                      # 90 x 100 x 120
    M, T = int(dens * 90 * 100 * 120), 65536
    x = _pts(rng, M)
    for wide in (False, True):
        c, f = _cplx(rng, M), _cplx(rng, N)
        if wide:
            c *= np.exp(4 * rng.standard_normal(M)).astype(np.float32)
            f *= np.exp(4 * rng.standard_normal(N)).astype(np.float32)
        e1, e2 = _sums64(x, c, f, N, T)
        p, g = mn.Type1PlanND(x, N, eps=eps), mn.Type2PlanND(x, N, eps=eps)
        assert p.n_up == [90, 100, 120] and p._store() is not None and g._store() is not None
        r = [float((a.to(torch.complex128) - b).norm() / b.norm()) for a, b in
             ((p.execute(c, return_np=False), e1), (g.execute(f, return_np=False)[:T], e2))]
        print(f"  wide={wide} type 1 {r[0]:.3e} type 2 {r[1]:.3e}", flush=True)
        assert max(r) <= most


def test_extents_leave_dense_sets_to_fp64_sums(mn):
    """fp32 sums lose to the tiles' fp64 ones where a cell sums many points
    (7.7e-7 against 7.0e-7 at 20 a cell, w = 8), so from 8 a cell on the tiles
    have them, on re-pointing as on a new plan; a plan built on them is one of
    tiles for good, as it would build two point states for every set."""
    print("case extents dense", flush=True)
    rng = np.random.default_rng(37)
    N, cells = (45, 50, 55), 90 * 100 * 120
    thin, dense = _pts(rng, 6 * cells), _pts(rng, 12 * cells)
    for first, kinds in ((thin, ("tiles", "zsweep")), (dense, ("tiles", "tiles"))):
        p = mn.Type1PlanND(first, N, eps=1e-7)
        assert p.pts.kind == kinds[1]
        for x, kind in zip((dense, thin), kinds):
            p.set_sources(x)
            assert p.pts.kind == kind and (p._store() is None) == (kind == "tiles")


def test_repointing_weighs_both_point_states(mn):
    """Moderately crowded sets, which the tiles would only just spread faster,
    stay with the sweep on re-pointing: the step pays for the tiles' point
    state too. Plans built on them take the tiles."""
    print("case repoint setup", flush=True)
    rng = np.random.default_rng(39)

    def radial(M, dim):
        v = rng.standard_normal((dim, M // 256 + 1, 1))
        v = v / np.linalg.norm(v, axis=0) * np.linspace(-np.pi, np.pi, 256, endpoint=False)
        return tuple(np.ascontiguousarray(a.reshape(-1)[:M]) for a in v)

    for N, M, eps, sweep, later in (((1024, 1024), 300_000, 1e-6, "ymfma", "ymfma"),
                                    ((45, 50, 55), 30_000, 1e-2, "zsweep", "tiles")):
        x = radial(M, len(N))
        p = mn.Type1PlanND(x, N, eps=eps)
        assert p.pts.kind == "tiles"
        p.set_sources(x)
        assert p.pts.kind == later
        p = mn.Type1PlanND(_pts(rng, M)[:len(N)], N, eps=eps)
        p.set_sources(x)
        assert p.pts.kind == sweep
        c = _cplx(rng, M)
        ref = mn.Type1PlanND(x, N, eps=eps, spread_method="gm").execute(c)
        assert np.linalg.norm(p.execute(c) - ref) <= 3e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("N,M,sweep", [((32, 32, 32), 1 << 18, "zsweep"),
                                       ((128, 128), 1 << 17, "ymfma")])
def test_native_route_depends_on_first_and_current_set_only(N, M, sweep, mn):
    """On the sweeps' own grids a plan built on crowded points looks at every
    set, also after ones that were spread out; a plan built on others, few
    points among them, reads nothing back and stays with the sweep. Results
    are those of the tiles."""
    print(f"case native route N={N}", flush=True)
    rng = np.random.default_rng(38)
    dim = len(N)
    dev = lambda x: tuple(torch.from_numpy(v).cuda() for v in x)
    crowd = dev([rng.uniform(0.1, 0.2, M) for _ in range(dim)])
    wide = dev([rng.uniform(-np.pi, np.pi, M) for _ in range(dim)])
    few = tuple(v[:1000].contiguous() for v in wide)
    c = _cplx(rng, M)
    ref = {k: mn.Type1PlanND(x, N, eps=1e-6, spread_method="gm").execute(c)
           for k, x in (("crowd", crowd), ("wide", wide))}

    # a sweep adds a cell's points one after another in fp32: each of the M
    # additions to the crowd's few cells rounds by up to 2^-24 of a partial sum
    # that grows as its root, sqrt(M / 2) 2^-24 of the whole in all
    swept = 2.0 ** -24 * np.sqrt(M / 2)

    def check(p, key):
        a = p.execute(c)
        tol = 3e-6 if key == "wide" or p.pts.kind == "tiles" else swept
        assert np.linalg.norm(a - ref[key]) <= tol * np.linalg.norm(ref[key])

    p = mn.Type1PlanND(crowd, N, eps=1e-6)
    for key, x, kind in (("wide", wide, sweep), ("crowd", crowd, "tiles"), ("wide", wide, sweep)):
        p.set_sources(x)
        assert p.pts.kind == kind
        check(p, key)
    for first in (wide, few):
        p = mn.Type1PlanND(first, N, eps=1e-6)
        torch.cuda.set_sync_debug_mode("error")
        try:
            p.set_sources(crowd)
        finally:
            torch.cuda.set_sync_debug_mode("default")
        assert p.pts.kind == sweep
        check(p, "crowd")


def test_route_follows_number_of_points(mn):
    """Re-pointing to another number of points takes the tiles and the route of
    a plan built on so many: the VALU y-sweep's grids go to the tiles from 2^17
    points on, the tiles' bins follow the points per cell."""
    print("case route by count", flush=True)
    rng = np.random.default_rng(40)
    pts = lambda M: tuple(rng.uniform(-np.pi, np.pi, M) for _ in range(2))
    for N, sizes, kinds in (((128, 135), (2000, 1 << 17, 2000), ("ysweep", "tiles", "ysweep")),
                            ((125, 135), (2000, 60000, 2000), ("tiles",) * 3)):
        p = mn.Type1PlanND(pts(sizes[-1]), N, eps=1e-6)
        for M, kind in zip(sizes, kinds):
            x, c = pts(M), _cplx(rng, M)
            p.set_sources(x)
            q = mn.Type1PlanND(x, N, eps=1e-6)
            assert p.pts.kind == q.pts.kind == kind
            assert list(p.pts.bins.m) == list(q.pts.bins.m)
            ref = q.execute(c)
            assert np.linalg.norm(p.execute(c) - ref) <= 1e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("N,M,crowded,kind", [((128, 135), 1 << 17, False, "ysweep"),
                                              ((128, 128), 1 << 17, True, "ymfma"),
                                              ((32, 32, 32), 1 << 18, True, "zsweep"),
                                              ((27, 25, 33), 20000, False, "zsweep")])
def test_step_under_capture(N, M, crowded, kind, mn):
    """A step (set_sources and execute) captured into a graph: nothing can be
    read back there, so the sweep takes the set where the grid has one; every
    replay equals the eager tiles, with eager work in between."""
    print(f"case capture N={N}", flush=True)
    rng = np.random.default_rng(41)
    dim = len(N)
    wide = [[rng.uniform(-np.pi, np.pi, M) for _ in range(dim)] for _ in range(3)]
    first = [rng.uniform(0.1, 0.2, M) for _ in range(dim)] if crowded else wide[0]
    x = [torch.from_numpy(v.copy()).cuda() for v in wide[0]]
    c = torch.from_numpy(_cplx(rng, M)).cuda()
    p = mn.Type1PlanND([torch.from_numpy(v).cuda() for v in first], N, eps=1e-6)
    p.set_sources(x)
    p.execute(c, return_np=False)       # tables and buffers
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        p.set_sources(x)
        out = p.execute(c, return_np=False)
    assert p.pts.kind == kind
    for w in wide:
        for d in range(dim):
            x[d].copy_(torch.from_numpy(w[d]))
        graph.replay()
        got = out.cpu().numpy()
        ref = mn.Type1PlanND(tuple(w), N, eps=1e-6, spread_method="gm").execute(c)
        assert np.linalg.norm(got - ref) <= 3e-6 * np.linalg.norm(ref)


@pytest.mark.parametrize("N,M,kind", [((32, 32, 32), 1 << 18, "zsweep"),
                                      ((128, 128), 1 << 17, "ymfma"),
                                      ((128, 135), 1 << 17, "ysweep")])
def test_od_keeps_the_sweep(N, M, kind, mn):
    """spread_method="od" keeps crowded and dense sets on the owner-computes
    sweeps, whose results repeat bit for bit."""
    print(f"case od N={N}", flush=True)
    rng = np.random.default_rng(42)
    x = tuple(rng.uniform(0.1, 0.2, M) for _ in N)
    c = _cplx(rng, M)
    p = mn.Type1PlanND(x, N, eps=1e-6, spread_method="od")
    assert p.pts.kind == kind and mn.Type1PlanND(x, N, eps=1e-6).pts.kind == "tiles"
    one = p.execute(c)
    assert np.array_equal(p.execute(c), one)
    p.set_sources(x)
    assert p.pts.kind == kind and np.array_equal(p.execute(c), one)


def test_crowding_rule_2d_near_break_even(mn):
    """Radial points on 2048^2, w = 7: 2^17 stay with the sweep (99 us against
    125 with the tiles), 3e5 leave it (153 against 130)."""
    print("case crowding rule 2d", flush=True)
    rng = np.random.default_rng(43)
    for M, kind in ((1 << 17, "ymfma"), (300_000, "tiles")):
        per = int(np.sqrt(M))
        v = rng.standard_normal((2, M // per + 1, 1))
        v = v / np.linalg.norm(v, axis=0) * np.linspace(-np.pi, np.pi, per, endpoint=False)
        x = tuple(np.ascontiguousarray(a.reshape(-1)[:M]) for a in v)
        assert mn.Type1PlanND(x, (1024, 1024), eps=1e-6).pts.kind == kind


def test_dense_narrow_kernels_on_extents(mn):
    """Up to w = 4 dense sets on small grids stored with extents go to the tiles
    by their number, on re-pointing as on a new plan."""
    print("case dense narrow extents", flush=True)
    rng = np.random.default_rng(44)
    N, cells = (25, 80, 36), 50 * 160 * 72
    thin, dense = _pts(rng, cells // 4), _pts(rng, cells)
    for eps, kind in ((1e-3, "tiles"), (1e-4, "zsweep")):
        p = mn.Type1PlanND(dense, N, eps=eps)
        assert p.n_up == [50, 160, 72] and p.pts.kind == kind
        for x, k in ((thin, "zsweep"), (dense, kind)):
            p.set_sources(x)
            assert p.pts.kind == k and (p._store() is None) == (k == "tiles")
            c = _cplx(rng, x[0].size)
            ref = mn.Type1PlanND(x, N, eps=eps, spread_method="gm").execute(c)
            assert np.linalg.norm(p.execute(c) - ref) <= 3e-6 * np.linalg.norm(ref)
