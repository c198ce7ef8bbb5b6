"""The type-1 tile spreads on the matrix cores (2D and 3D, bins of 17 - w)
against the fp64 oracle's spread of the same cells and fractions: the widths at
both ends, grids smaller than a tile, partial and wrapping bins, crowded
points (many subproblems of one bin), and batches."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,N,eps,M,B,crowd", [
    (2, (5, 6), 1e-5, 300, 1, False), (2, (33, 21), 1e-4, 2000, 1, False),
    (2, (33, 21), 1e-6, 5000, 3, True), (2, (61, 50), 1e-11, 7000, 2, False),
    (2, (16, 17), 1e-13, 2000, 1, False),
    (3, (5, 6, 7), 1e-4, 1, 1, False), (3, (13, 9, 11), 1e-4, 4000, 1, False),
    (3, (13, 9, 11), 1e-6, 5000, 3, True), (3, (19, 18, 17), 1e-9, 2000, 1, False),
    (3, (17, 16, 18), 1e-15, 70, 2, False),
])
def test_tile_spread_vs_oracle(dim, N, eps, M, B, crowd, oracle, mn):
    from mlx_nufft_amd import _engine as E

    print(f"case tile spread dim={dim} N={N} eps={eps} M={M} B={B} crowd={crowd}", flush=True)
    rng = np.random.default_rng(21)
    x = [rng.uniform(-0.1, 0.1, M) if crowd else rng.uniform(-np.pi, np.pi, M)
         for _ in range(dim)]
    c = (rng.standard_normal((B, M)) + 1j * rng.standard_normal((B, M))).astype(np.complex64)
    p = mn.Type1PlanND(tuple(x), N, eps=eps, spread_method="gm")
    assert p.pts.kind == "tiles" and max(p.bins.m[d] + p.w - 1 for d in range(dim)) <= 16
    cd = torch.from_numpy(c).cuda()
    grids = torch.empty((B, *p.n_up), dtype=torch.complex64, device="cuda")
    E.spread_batch(p.pts, p.beta, cd, grids)
    one = torch.empty(p.n_up, dtype=torch.complex64, device="cuda")
    E.spread(p.pts, p.beta, cd[0], one)
    i1, fr = oracle.setpts_t12(x, p.n_up, p.w)
    # fp32 weights: a few ulp (2^-24) of exponent error times beta <= 37 per
    # axis; the sums are fp64 until the fp32 flush
    tol = dim * 4 * 2.0 ** -24 * max(8.0, p.beta)
    for b in range(B):
        ref = oracle.spread(i1, fr, c[b], p.n_up, p.w, p.beta)
        assert oracle.rel_l2(grids[b].cpu().numpy(), ref) < tol
    assert oracle.rel_l2(one.cpu().numpy(), grids[0].cpu().numpy()) < 1e-6


@pytest.mark.parametrize("M", [9203, 100_000])
def test_small_upsampling_no_less_precise_than_lds_tiles(M, mn, monkeypatch):
    """At sigma = 1.25 the deconvolution magnifies the rounding of the fp32
    sums that join subproblems: the matrix-core tiles are no further from 64
    bits there than the LDS tiles of 1024 points a subproblem (over four sets;
    5 % of slack for the order of the atomics), whole and by disjoint groups."""
    print(f"case sigma 1.25 tiles M={M}", flush=True)
    rng = np.random.default_rng(22)
    N, eps = (13, 21, 19), 1e-5                           # 18 x 30 x 24, w = 9
    ks = [torch.arange(-(n // 2), n - n // 2, dtype=torch.float64, device="cuda") for n in N]
    sums = {"mfma": 0.0, "groups": 0.0, "lds": 0.0}
    for _ in range(4):
        x = tuple(torch.from_numpy(rng.uniform(-np.pi, np.pi, M)).cuda() for _ in range(3))
        c = torch.from_numpy((rng.standard_normal(M) + 1j * rng.standard_normal(M))
                             .astype(np.complex64)).cuda()
        exact = torch.zeros(N[0] * N[1], N[2], dtype=torch.complex128, device="cuda")
        for lo in range(0, M, 8192):
            e = [torch.polar(torch.ones_like(p), p) for p in
                 (x[d][lo:lo + 8192, None] * ks[d] for d in range(3))]
            xy = (e[0][:, :, None] * (c[lo:lo + 8192, None] * e[1])[:, None, :])
            exact += xy.reshape(-1, N[0] * N[1]).T.contiguous() @ e[2]
        exact = exact.reshape(N)
        monkeypatch.delenv("MN_BIN_M", raising=False)
        p = mn.Type1PlanND(x, N, eps=eps, upsampfac=1.25)
        monkeypatch.setenv("MN_BIN_M", "9")
        q = mn.Type1PlanND(x, N, eps=eps, upsampfac=1.25)
        assert p.pts.kind == q.pts.kind == "tiles" and (p.bins.m[0], q.bins.m[0]) == (8, 9)
        none = torch.zeros(M, dtype=torch.int64, device="cuda")
        for k, f in (("mfma", p.execute(c, return_np=False)),
                     ("groups", p.execute_disjoint(c, none, return_np=False)[0]),
                     ("lds", q.execute(c, return_np=False))):
            sums[k] += float((f.to(torch.complex128) - exact).norm() / exact.norm()) / 4
    print("  " + ", ".join(f"{k} {v:.3e}" for k, v in sums.items()))
    assert max(sums["mfma"], sums["groups"]) <= 1.05 * sums["lds"]
