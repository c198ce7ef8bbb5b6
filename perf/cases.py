"""The work that programs have this engine do, as cases that can be timed.

A case is a dict of plain values:
  call   "oneshot"  a finufft-style function on numpy arrays (plan, run, copy back)
         "t1"       Type1PlanND.execute (or execute_batch for B > 1), plan kept
         "t2"       Type2PlanND.execute, plan kept
         "both"     type 2 then type 1 at the same points, plans kept: one
                    gradient of an iterative reconstruction
         "step"     Type1PlanND.set_sources with the step's points, then execute
         "t3"       Type3Plan.execute, plan kept
  dim, M (points), N0..N2 (modes), eps, sigma (upsampfac), B (vectors),
  points "uniform" or "radial" (spokes through the origin); type 3 instead has
  P sources in [-X, X]^3 and M targets in [-S, S]^3.

listed() names the cases, draw() gives further ones of the same ranges.
exact() evaluates a case in 64 bits with plain torch and numpy.
"""

import math

import numpy as np
import torch

import mlx_nufft_amd as mn


def _case(name, call, dim, M, N, eps, sigma=2.0, B=1, points="uniform"):
    c = {"name": name, "call": call, "dim": dim, "M": M, "eps": eps, "sigma": sigma, "B": B,
         "points": points}
    for d in range(dim):
        c[f"N{d}"] = N[d]
    return c


def _case3(name, P, M, X, S, eps):
    return {"name": name, "call": "t3", "dim": 3, "P": P, "M": M, "X": X, "S": S, "eps": eps}


def listed():
    return [
        # a script's single small transform on host arrays: latency of the whole call
        _case("oneshot 2d small", "oneshot", 2, 3000, (40, 36), 1e-6),
        # a spectrum of 1e5 unevenly sampled values (the benchmark's 1D size)
        _case("1d type 1", "t1", 1, 100_000, (4096,), 1e-6),
        # resampling a long ragged record at scattered times
        _case("1d type 2 long", "t2", 1, 3_000_000, (500_001,), 1e-6),
        # eight coils or channels over one point set (the benchmark's batched 2D size)
        _case("2d type 1 x 8", "t1", 2, 10_000_000, (1024, 1024), 1e-6, B=8),
        # radial MRI forward model: 512 spokes of 2048 samples (the benchmark's)
        _case("2d type 2 radial", "t2", 2, 512 * 2048, (1024, 1024), 1e-6, points="radial"),
        # one gradient of a 2D reconstruction on an odd field of view
        _case("2d both ragged", "both", 2, 2_000_000, (601, 443), 1e-5),
        # moving particles: new points and a transform per step (the headline benchmark)
        _case("3d step", "step", 3, 20_000_000, (256, 256, 256), 1e-5),
        # its adjoint: field values back at the particles
        _case("3d type 2", "t2", 3, 20_000_000, (256, 256, 256), 1e-5),
        # one gradient of a 3D reconstruction on a ragged box
        _case("3d both ragged", "both", 3, 2_000_000, (135, 111, 90), 1e-6),
        # the same with the small upsampling factor (wide kernel, small grid)
        _case("3d both sigma 1.25", "both", 3, 1_000_000, (128, 128, 128), 1e-5, sigma=1.25),
        # type 3 between two point clouds (the benchmark's two geometries)
        _case3("3d type 3 compact", 1_000_000, 1_000_000, 1.0, 200.0, 1e-5),
        _case3("3d type 3 wide", 1_000_000, 512 * 512, 30.0, 20.0, 3e-5),
    ]


_TAPS = 1.5e9     # points x taps x vectors of a drawn case, at most
_CELLS = 1.3e8    # fine-grid cells x vectors of a drawn case, at most


def _log(rng, lo, hi):
    return math.exp(rng.uniform(math.log(lo), math.log(hi)))


def draw(rng):
    call = rng.choice(["oneshot", "t1", "t1", "t2", "t2", "both", "both", "step", "t3"])
    eps = rng.choice([1e-3, 1e-4, 1e-5, 1e-5, 1e-6, 1e-6])
    if call == "t3":
        P, M = int(_log(rng, 3e4, 1e6)), int(_log(rng, 3e4, 1e6))
        X = _log(rng, 0.5, 30.0)
        S = min(_log(rng, 60.0, 600.0) / X, 300.0)
        return {"call": "t3", "dim": 3, "P": P, "M": M, "X": round(X, 4), "S": round(S, 4),
                "eps": max(eps, 1e-5)}
    dim = rng.choice([1, 2, 2, 3, 3])
    sigma = rng.choice([2.0, 2.0, 2.0, 2.0, 1.25])
    B = rng.choice([2, 3, 4, 8]) if call == "t1" and rng.random() < 0.4 else 1
    w = mn.kernel_params(eps, sigma)[0]
    top = min(1e7, _TAPS / (w ** dim * B))
    if call == "oneshot":
        M = _log(rng, 300, 3e5)
    else:
        M = _log(rng, 3e4, top)
    cells = min(_CELLS / B, 2e7 if call == "oneshot" else _CELLS)
    modes = min(max(_log(rng, M / 20, M * 20), 4.0 ** dim * 8), cells / (1.15 * sigma) ** dim)
    if dim == 1:
        modes = min(modes, 4e6)
    side = modes ** (1.0 / dim)
    N = [max(4, int(side * _log(rng, 0.7, 1.4))) for _ in range(dim)]
    while math.prod(N) * (1.15 * sigma) ** dim > cells:
        N = [max(4, int(n * 0.9)) for n in N]
    points = "radial" if dim > 1 and rng.random() < 0.3 else "uniform"
    c = _case("", call, dim, int(M), N, eps, sigma, B, points)
    del c["name"]
    return c


# ---------------------------------------------------------------------------
# inputs


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(1_000_003 * (seed + 1))
    return g


def _uniform(g, n, lo, hi):
    return lo + (hi - lo) * torch.rand(n, dtype=torch.float64, device="cuda", generator=g)


def _cplx(g, *shape):
    return torch.randn(*shape, dtype=torch.complex64, device="cuda", generator=g)


def _points(case, g):
    dim, M = case["dim"], case["M"]
    if case["points"] == "uniform":
        return tuple(_uniform(g, M, -math.pi, math.pi) for _ in range(dim))
    # spokes of evenly spaced radii at random angles, through the origin
    per = min(2048, max(16, int(math.sqrt(M))))
    spokes = -(-M // per)
    r = -math.pi + 2.0 * math.pi / per * torch.arange(per, dtype=torch.float64, device="cuda")
    v = torch.randn(dim, spokes, dtype=torch.float64, device="cuda", generator=g)
    v = v / v.norm(dim=0, keepdim=True)
    return tuple((v[d][:, None] * r[None, :]).reshape(-1)[:M].contiguous() for d in range(dim))


def _modes(case):
    return tuple(case[f"N{d}"] for d in range(case["dim"]))


def _inputs(case, seed):
    """(points, strengths or None, modes or None), or for type 3 (sources, strengths, targets)."""
    g = _gen(seed)
    if case["call"] == "t3":
        x = tuple(_uniform(g, case["P"], -case["X"], case["X"]) for _ in range(3))
        c = _cplx(g, case["P"])
        return x, c, tuple(_uniform(g, case["M"], -case["S"], case["S"]) for _ in range(3))
    x = _points(case, g)
    c = f = None
    if case["call"] != "t2":
        c = _cplx(g, case["B"], case["M"]) if case["B"] > 1 else _cplx(g, case["M"])
    if case["call"] in ("t2", "both"):
        f = _cplx(g, *_modes(case))
    return x, c, f


def prepare(case, seed):
    x, c, f = _inputs(case, seed)
    if case["call"] == "t3":
        return {"call": "t3", "c": c, "plan": mn.Type3Plan(x, f, eps=case["eps"])}
    N, kw = _modes(case), {"eps": case["eps"], "upsampfac": case["sigma"]}
    s = {"call": case["call"], "dim": case["dim"], "N": N, "c": c, "f": f, "kw": kw}
    if case["call"] == "oneshot":
        s["x"] = tuple(v.cpu().numpy() for v in x)
        s["c"] = c.cpu().numpy()
        return s
    if case["call"] == "step":
        s["x"] = x
    if case["call"] != "t2":
        s["t1"] = mn.Type1PlanND(x, N, isign=+1, **kw)
    if case["call"] in ("t2", "both"):
        s["t2"] = mn.Type2PlanND(x, N, isign=-1, **kw)
    return s


def run(s):
    call = s["call"]
    if call == "t3":
        return s["plan"].execute(s["c"], return_np=False)
    if call == "oneshot":
        fn = (mn.nufft1d1, mn.nufft2d1, mn.nufft3d1)[s["dim"] - 1]
        return fn(*s["x"], s["c"], s["N"], **s["kw"])
    if call == "step":
        s["t1"].set_sources(s["x"])
        return s["t1"].execute(s["c"], return_np=False)
    if call == "t1":
        if s["c"].dim() == 2:
            return s["t1"].execute_batch(s["c"], return_np=False)
        return s["t1"].execute(s["c"], return_np=False)
    if call == "t2":
        return s["t2"].execute(s["f"], return_np=False)
    return (s["t2"].execute(s["f"], return_np=False), s["t1"].execute(s["c"], return_np=False))


# ---------------------------------------------------------------------------
# what a pass cannot do without


def work(case):
    """Bytes: each point's position, strength and mode once. Operations: the
    kernel's taps and the pruned transform's share of 5 n log2 n."""
    eps, dim = case["eps"], case["dim"]
    if case["call"] == "t3":
        w = mn.kernel_params(eps, 1.25)[0]
        n = [1.25 * (2.5 * case["S"] * case["X"] / math.pi + w + 1)] * 3
        points = case["P"] + case["M"]
        fft = 5 * math.prod(n) * sum(math.log2(v) for v in n)
        return {"bytes": points * (24 + 8 + 8), "flops": 4 * points * w ** 3 + fft}
    w = mn.kernel_params(eps, case["sigma"])[0]
    N, B, M = _modes(case), case["B"], case["M"]
    ways = 2 if case["call"] == "both" else 1
    pos = 8 * dim  # fp64 coordinates, or a kept 32-bit cell and fraction, per dim
    n = [case["sigma"] * v for v in N]
    fft = 0.0
    for d in range(dim):  # lines of axis d: full before it, pruned after it
        fft += 5 * math.prod(n[:d + 1]) * math.prod(N[d + 1:]) * math.log2(max(2.0, n[d]))
    return {"bytes": ways * (M * pos + B * 8 * (M + math.prod(N))),
            "flops": ways * B * (4 * M * w ** dim + fft)}


def tolerance(case):
    """Four times what the same path was seen to differ by with its sums in
    another order (tiles instead of sweeps, full instead of pruned transform;
    in type 3 the gather along another axis): 32-bit weights, sums and
    transforms give 4e-7 at most in the cases tried, and points crowded at a
    centre are allowed twice that. The modes at the edge of the box are divided
    by the kernel's small transform there, which at upsampling 1.25 raises that
    rounding to 3.2e-5 (3.1e-3 of a single value) and in type 3 to 2.5e-6."""
    if case["call"] == "t3":
        return {"rel": 1e-5}
    if case["sigma"] != 2.0:
        return {"rel": 1.3e-4, "max": 0.015}
    return {"rel": 3e-6}


# ---------------------------------------------------------------------------
# 64 bits: direct sums for type 3, and for types 1 and 2 a transform with a
# 13-point kernel at upsampling 2, whose own error is below 1e-11

_W, _BETA = 13, 2.30 * 13
_LIMIT = 8e9     # point x tap pairs, about 20 s
_PAIRS = 3.2e11  # source x target pairs of a direct sum


def _es64(t):
    z = torch.clamp(1.0 - (2.0 / _W * t) ** 2, min=0.0)
    return torch.exp(_BETA * (torch.sqrt(z) - 1.0))


def _grid64(n):
    n = max(2 * n, 2 * _W)
    n += n & 1
    while True:
        r = n
        for p in (2, 3, 5):
            while r % p == 0:
                r //= p
        if r == 1:
            return n
        n += 2


def _dec64(N, n):
    t, wt = np.polynomial.legendre.leggauss(160)
    dq = 0.5 * (t + 1.0) * (_W / 2.0)
    fq = wt * (_W / 4.0) * np.exp(_BETA * (np.sqrt(1.0 - (2.0 * dq / _W) ** 2) - 1.0))
    k = np.arange(-(N // 2), N - N // 2, dtype=np.float64)
    out = np.empty(N)
    for a in range(0, N, 65536):
        out[a:a + 65536] = 0.5 / (fq @ np.cos(np.outer(dq, 2.0 * np.pi * k[a:a + 65536] / n)))
    return torch.from_numpy(out).cuda()


def _taps(x, n, dim, lo, hi):
    """Flat grid indices and weights (m, W^dim) of points [lo, hi)."""
    idx = wt = None
    for d in range(dim):
        X = torch.remainder(x[d][lo:hi], 2.0 * math.pi) * (n[d] / (2.0 * math.pi))
        i0 = torch.ceil(X - _W / 2.0)
        t = i0[:, None] + torch.arange(_W, device="cuda", dtype=torch.float64)
        wd = _es64(t - X[:, None])
        td = torch.remainder(t.long(), n[d])
        if idx is None:
            idx, wt = td, wd
        else:
            idx = (idx[:, :, None] * n[d] + td[:, None, :]).reshape(hi - lo, -1)
            wt = (wt[:, :, None] * wd[:, None, :]).reshape(hi - lo, -1)
    return idx, wt


def _chunks(M, dim):
    step = max(1, (1 << 26) // _W ** dim)
    return [(lo, min(M, lo + step)) for lo in range(0, M, step)]


def _ks(N, n):
    k = torch.arange(-(N // 2), N - N // 2, device="cuda")
    return torch.remainder(k, n)


def _type1_64(x, c, N, isign):
    dim, n = len(N), [_grid64(v) for v in N]
    grid = torch.zeros(2, math.prod(n), dtype=torch.float64, device="cuda")
    for lo, hi in _chunks(x[0].numel(), dim):
        idx, wt = _taps(x, n, dim, lo, hi)
        idx = idx.reshape(-1)
        cc = c[lo:hi].to(torch.complex128)
        grid[0].index_add_(0, idx, (wt * cc.real[:, None]).reshape(-1))
        grid[1].index_add_(0, idx, (wt * cc.imag[:, None]).reshape(-1))
    F = torch.complex(grid[0], grid[1]).reshape(n)
    del grid
    for d in range(dim - 1, -1, -1):
        F = torch.fft.ifft(F, dim=d, norm="forward") if isign > 0 else torch.fft.fft(F, dim=d)
        F = F.index_select(d, _ks(N[d], n[d]))
        F = F * _dec64(N[d], n[d]).reshape([-1 if e == d else 1 for e in range(dim)])
    return F


def _type2_64(x, f, N, isign):
    dim, n = len(N), [_grid64(v) for v in N]
    F = f.to(torch.complex128)
    for d in range(dim):
        F = F * _dec64(N[d], n[d]).reshape([-1 if e == d else 1 for e in range(dim)])
        shape = list(F.shape)
        shape[d] = n[d]
        G = torch.zeros(shape, dtype=torch.complex128, device="cuda")
        G.index_copy_(d, _ks(N[d], n[d]), F)
        F = torch.fft.ifft(G, dim=d, norm="forward") if isign > 0 else torch.fft.fft(G, dim=d)
        del G
    F = F.reshape(-1)
    out = torch.empty(x[0].numel(), dtype=torch.complex128, device="cuda")
    for lo, hi in _chunks(out.numel(), dim):
        idx, wt = _taps(x, n, dim, lo, hi)
        out[lo:hi] = (F[idx] * wt).sum(dim=1)
    return out


def _type3_64(x, c, s):
    xs, cc = torch.stack(x), c.to(torch.complex128)
    M = s[0].numel()
    out = torch.empty(M, dtype=torch.complex128, device="cuda")
    step = max(1, (1 << 27) // xs.shape[1])
    for lo in range(0, M, step):
        hi = min(M, lo + step)
        ph = s[0][lo:hi, None] * xs[0] + s[1][lo:hi, None] * xs[1] + s[2][lo:hi, None] * xs[2]
        co, si = torch.cos(ph), torch.sin_(ph)
        re = co @ cc.real - si @ cc.imag
        out[lo:hi] = torch.complex(re, co @ cc.imag + si @ cc.real)
    return out


def exact(case, seed):
    x, c, f = _inputs(case, seed)
    if case["call"] == "t3":
        if case["P"] * case["M"] > _PAIRS:
            return None
        return _type3_64(x, c, f)
    N, B, M, dim = _modes(case), case["B"], case["M"], case["dim"]
    ways = 2 if case["call"] == "both" else 1
    if M * B * ways * _W ** dim > _LIMIT:
        return None
    if case["call"] == "t2":
        return _type2_64(x, f, N, -1)
    if B > 1:
        return torch.stack([_type1_64(x, c[b], N, +1) for b in range(B)])
    t1 = _type1_64(x, c, N, +1)
    if case["call"] == "both":
        return (_type2_64(x, f, N, -1), t1)
    return t1.cpu().numpy() if case["call"] == "oneshot" else t1
