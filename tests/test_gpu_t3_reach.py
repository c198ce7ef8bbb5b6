"""Line passes over a part of their lines and outputs, and the part of the
type-3 inner grid that targets reach.

A partial pass runs the same operations on the lines it keeps, so it equals
the whole pass bit for bit there and writes nothing elsewhere."""

import numpy as np
import pytest
import torch

from mlx_nufft_amd import _engine as E


@pytest.mark.parametrize("n,w", [(32, 8), (75, 9), (225, 9), (640, 8), (18, 9), (25, 2)])
def test_target_cells_hold_every_tap(n, w):
    """[lo, hi) holds ceil(lam - w/2) + (0 .. w - 1) for lam = n/2 +- R, or is
    the whole axis where such a tap would wrap."""
    for R in np.linspace(0.0, 0.5 * n, 41):
        lo, hi = E.target_cells(n, w, R)
        assert 0 <= lo < hi <= n
        lam = 0.5 * n + np.linspace(-R, R, 101)
        first = np.ceil(lam - 0.5 * w)
        inside = first.min() >= lo and first.max() + w <= hi
        assert inside or (lo, hi) == (0, n)


# (A, nin, B, n, layout, keep, (period, q, c))
PARTS = [
    (5, 19, 24, 30, "anb", (8, 24), (24, (0, 5), (8, 24))),        # y pass
    (3, 180, 225, 225, "anb", (16, 208), (225, (0, 3), (16, 208))),  # odd B
    (1, 12, 20 * 18, 18, "lines_first", (1, 17), (18, (3, 19), (2, 17))),  # x pass, odd part
    (1, 12, 20 * 16, 18, "lines_first", (0, 18), (16, (4, 20), (0, 16))),  # whole rows
    (6 * 10, 40, 1, 50, "anb", (8, 41), (10, (1, 5), (0, 10))),    # contiguous, whole rows
    (6 * 10, 40, 1, 50, "anb", (8, 41), (10, (1, 5), (3, 8))),     # contiguous, part of rows
    (33, 40, 1, 50, "lines_last", (9, 10), None),
    (3 * 5, 4000, 1, 5000, "anb", (401, 4600), (5, (1, 3), (1, 4))),  # long lines
    (2, 30, 12, 36, "anb", (4, 32), None),
]


@pytest.mark.gpu
@pytest.mark.parametrize("c64", [False, True])
@pytest.mark.parametrize("A,nin,B,n,layout,keep,rows", PARTS)
def test_partial_pass_equals_whole_pass(A, nin, B, n, layout, keep, rows, c64):
    print(f"case part A={A} nin={nin} B={B} n={n} {layout} {keep} {rows} c64={c64}", flush=True)
    dt = torch.complex64 if c64 else torch.complex128
    x = torch.randn(A, nin, B, dtype=torch.complex128, device="cuda")
    dec = torch.rand(nin, dtype=torch.float64, device="cuda")
    whole = torch.empty(A * B * n, dtype=dt, device="cuda")
    part = torch.full_like(whole, 7.0)
    E.fft64_lines(A, nin, B, n, +1, x, dec, whole, layout=layout)
    E.fft64_lines(A, nin, B, n, +1, x, dec, part, layout=layout, keep=keep, rows=rows)
    line = torch.zeros(A * B, dtype=torch.bool)
    if rows is None:
        line[:] = True
    else:
        period, q, c = rows
        line.view(-1, period)[q[0]:q[1], c[0]:c[1]] = True
    out = torch.zeros(n, dtype=torch.bool)
    out[keep[0]:keep[1]] = True
    if layout == "anb":
        kept = line.view(A, 1, B) & out.view(1, n, 1)
    elif layout == "lines_last":
        kept = out.view(n, 1) & line.view(1, -1)
    else:
        kept = line.view(-1, 1) & out.view(1, n)
    kept = kept.reshape(-1).cuda()
    assert torch.equal(part[kept], whole[kept])
    assert bool((part[~kept] == 7.0).all())


@pytest.mark.gpu
@pytest.mark.parametrize("X,S,M", [((1.0,) * 3, (90.0, 120.0, 9.0), 3000),
                                   ((1.0,) * 3, (80.0, 95.0, 60.0), 400_000),
                                   ((120.0, 1.0, 2.0), (12.0, 3.0, 4.0), 5000)])
def test_unreached_cells_do_not_matter(X, S, M):
    """With every cell NaN before the passes, results are those of the whole
    transform: tiles, direct gather and the reversed axis order. The spread's
    atomics may add in another order, 2^-53 of the sums each."""
    print(f"case reach X={X} S={S} M={M}", flush=True)
    import mlx_nufft_amd as mn

    rng = np.random.default_rng(5)
    x = tuple(rng.uniform(-a, a, 4000) for a in X)
    s = tuple(100.0 + rng.uniform(-a, a, M) for a in S)
    c = (rng.standard_normal(4000) + 1j * rng.standard_normal(4000)).astype(np.complex64)
    p = mn.Type3Plan(x, s, eps=1e-5)
    assert any(r != (0, n) for r, n in zip(p._reach, p.n_up))
    for t in (p._buffers()[1], *p._T):
        t.fill_(float("nan"))
    part = p.execute(c)
    p._reach = [(0, n) for n in p.n_up]
    whole = p.execute(c)
    assert np.isfinite(part).all()
    assert np.abs(part - whole).max() <= 1e-6 * np.abs(whole).max()
