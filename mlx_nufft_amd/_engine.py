"""Thin wrappers over the C-ABI used by the plan classes: point setup, the
stable bin sort, subproblem tables, spread/interp, deconvolution, FFT and
expi. Every function takes and returns torch device tensors and runs on the
current stream; shapes are validated by the C side as well.

Bin geometry (the tile a workgroup owns) is chosen here, per dim and kernel
width, from the LDS budget of one CDNA4 workgroup.
"""

import contextlib
import ctypes
import math
import os

import numpy as np
import torch

from . import _lib as L

_require = L.require

MSUB = 1024                 # max points per spread/interp subproblem
TILE_BUDGET = 80 * 1024     # LDS bytes for one padded tile (2 workgroups/CU)


_budget = None


def tile_budget():
    """LDS bytes for one tile: TILE_BUDGET, capped by the device limit."""
    global _budget
    if _budget is None:
        try:
            dev = int(L.lib().mn_device_lds_bytes())
        except RuntimeError:
            dev = TILE_BUDGET
        _budget = min(TILE_BUDGET, dev if dev > 0 else 65536)
    return _budget


SPREAD_CELL_BYTES = 16   # spread tiles accumulate complex values in fp64
INTERP_CELL_BYTES = 8    # interp tiles hold complex64 grid values


def bin_sizes(dim, w, n_up, cell_bytes=SPREAD_CELL_BYTES, npts=None):
    """Bin size m per dim: the padded tile (m + w - 1 cells per dim,
    cell_bytes each) must fit tile_budget() bytes of LDS. npts (the number
    of points, when known) lets the 3D interp tiles grow for sparse points.
    Overridable with the environment variable MN_BIN_M="m0,m1,m2" (tuning)."""
    budget = tile_budget()
    env = os.environ.get("MN_BIN_M")
    if env:
        m = [int(v) for v in env.split(",")]
        m = (m + [m[-1]] * 3)[:dim]
    elif dim == 1:
        m = [1024]
    elif dim == 2:
        m = [32, 32]
    elif cell_bytes == INTERP_CELL_BYTES:
        # interp is bound by staging tiles: small bins keep about 9
        # workgroups resident per CU, which beats the smaller halo re-read of
        # big tiles (MI355X, 3D type 2 at 512^3: 2.0 ms at m = 8, 3.1 ms at
        # 16). Along z (the contiguous axis) the padded tile row is made 17
        # cells for w >= 5: rows of 16 (and 12) cells put the lane pairs'
        # LDS reads on conflicting banks. Type-2 execute, 2e7 points on
        # 512^3, m = (8, 8, m2): w = 5: 2.11 ms at m2 = 8, 1.94 at 13;
        # w = 6: 2.44 at 8, 2.35 at 12, 3.07 at 11; w = 7: 3.13 at 8, 3.03
        # at 11, 4.19 at 10. At w = 4, 8 is best within 2 %.
        # Sparse points (under 0.1 per cell, as type-3 targets) leave few
        # points per bin, so the tile load dominates and wider bins re-read
        # less halo: cfg 5's targets (1e6 on 240^3, w = 9) gather in 0.276 ms
        # with m = (11, 11, 9), 0.289 with 10^3, 0.318 with 9^3, 0.361 with
        # (8, 8, 9).
        mxy = 11 if (dim == 3 and npts is not None
                     and npts < 0.1 * float(np.prod([float(n) for n in n_up]))) else 8
        m = [mxy, mxy, max(8, 18 - w) if w >= 5 else 8]
    else:
        side = int(round((budget / cell_bytes) ** (1.0 / 3.0) - 1e-9))
        while cell_bytes * side ** 3 > budget:
            side -= 1
        m = [max(1, side - w + 1)] * 3
    m = [max(1, min(int(mi), int(n))) for mi, n in zip(m, n_up)]
    while cell_bytes * int(np.prod([mi + w - 1 for mi in m])) > budget and max(m) > 1:
        k = int(np.argmax(m))
        m[k] -= 1
    return m


def make_bins(dim, w, n_up, m=None, cell_bytes=SPREAD_CELL_BYTES, npts=None):
    if m is None:
        m = bin_sizes(dim, w, n_up, cell_bytes, npts=npts)
    return L.Bins.make(dim, w, list(n_up), m)


def spread_bins(dim, w, n_up, P):
    """Bins of the type-1 tile spread for about P points. Bins of 17 - w cells
    give padded tiles of at most 16 cells per dim, which are accumulated on the
    matrix cores; their work per point hardly depends on w, where LDS atomics
    cost w^dim, but smaller tiles flush more halo cells. So the matrix cores
    take 3D from w = 5 (us, LDS / matrix cores: 1e6 points on 200 x 180 x 160,
    w = 4: 191 / 219; on 240^3 7e3 to 1.4e6 points, w = 5: 110 / 57 to
    401 / 373, w = 7: 178 / 69 to 798 / 563, w = 12: 763 / 135 to 7928 / 3576;
    at w = 5 dense sets that are spread out pay for what crowded ones gain: 4
    points a cell on 50 x 30 x 180 282 / 324, but 5e6 radial ones on 256^3
    4629 / 1493)
    and 2D from w = 5 where the points fill the grid (2000^2, w = 6: 0.3
    points per cell 90 / 101, 0.6 143 / 101, 2.4 506 / 281; w = 12: 0.3
    272 / 387, 0.6 505 / 408); wider 2D kernels leave bins of 4 cells or fewer
    and need more. 3D kernels of 13 to 16 cells leave bins of 4 to 1, which are
    still the faster ones (120^3, 3e4 to 3e6 points: w = 13 1775 / 478 to
    12669 / 1337, w = 16 6704 / 1112 to 65124 / 55538), until there are so many
    of them that a launch of 256 threads for each that holds points would pass
    2^32, or their tables (24 bytes a bin) 3 GB. MN_BIN_M overrides the bins."""
    if dim == 1 or w <= 4 or os.environ.get("MN_BIN_M"):
        return make_bins(dim, w, n_up, cell_bytes=SPREAD_CELL_BYTES)
    if dim == 2:
        full = 0.4 if w <= 12 else 1.0
        if w > 14 or P < full * float(n_up[0]) * float(n_up[1]):
            return make_bins(dim, w, n_up, cell_bytes=SPREAD_CELL_BYTES)
    if dim == 3 and w == 5:
        # grids smaller than a tile, crowded: 137203 points on 12 x 20 x 10 105 us
        # with the matrix cores at best, 77 with LDS; 2e4 points 52 and 75
        cells = float(n_up[0]) * float(n_up[1]) * float(n_up[2])
        if cells < 4096 and P > 25 * cells:
            return make_bins(dim, w, n_up, cell_bytes=SPREAD_CELL_BYTES)
    bins = make_bins(dim, w, n_up, m=[max(1, min(17 - w, int(k))) for k in n_up])
    # subproblems: one for each bin with points, and one more for every 1024
    if bins.nbins > 1 << 27 or min(bins.nbins, P) + P // MSUB + MSUB >= 1 << 24:
        return make_bins(dim, w, n_up, cell_bytes=SPREAD_CELL_BYTES)
    return bins


def spread_msub(bins, P, sigma=2.0):
    """Points per subproblem of the type-1 tile spread: MSUB, but in steps of
    the matrix-core kernels' 64-point batches fewer where MSUB would leave the
    chip idle (2D tiles take one wave, 3D ones four): 1e4 points on
    18 x 24 x 30, w = 7, take 27 us instead of 100, 5e5 on 66 x 74 36 instead
    of 50; 5e5 points on 144 x 128 x 125 already fill it (more, smaller ones
    flush more tiles: 585 against 527 us for 4 vectors). The LDS kernels keep
    MSUB (1e5 points in 1D: 17 us, 19 to 25 with fewer), and so does sigma < 2
    from w = 8 on, whose deconvolution magnifies the rounding of the fp32 sums
    that join the subproblems: w = 9 at sigma = 1.25 on 18 x 30 x 24, 9e3 / 1e5
    points, 9.2e-6 / 1.22e-5 from 64 bits with short ones, 6.7e-6 / 8.1e-6 with
    MSUB and 7.3e-6 / 9.1e-6 in LDS tiles (47 / 76, 71 / 148 and 188 / 333 us);
    at w = 7 the kernel's own 9.9e-5 hides it. In 2D no cell takes the edges of
    more than 500 subproblems on average, or the atomics wait for each other:
    3 vectors of 63371 points on 10 x 36, w = 5, 63 us with 64, 39 with 128, of
    5e5 points 153 with 256, 88 to 108 with 512 and more (LDS tiles 50 and 99)."""
    dim, w = bins.dim, bins.w
    if (sigma < 2.0 and w >= 8) or dim == 1 or max(bins.m[d] + w - 1 for d in range(dim)) > 16:
        return MSUB
    least = 64
    if dim == 2:
        cells = float(bins.n[0]) * float(bins.n[1])
        least = max(64, math.ceil(P * 256 / (500.0 * cells) / 64) * 64)
    return min(MSUB, max(least, (P // (2048 if dim == 2 else 512) + 63) // 64 * 64))


def key_bits(bins):
    return max(1, int(bins.nbins - 1).bit_length())


def _rows(t, dim):
    return [t[d] for d in range(dim)]


def setpts_t12(bins, xs, prec64):
    """Cells, fractions and bin keys of type-1/2 points (caller order)."""
    dim, P = bins.dim, xs[0].numel()
    dev = xs[0].device
    i1 = torch.empty((dim, P), dtype=torch.int32, device=dev)
    fr = torch.empty((dim, P), dtype=torch.float32, device=dev)
    key = torch.empty(P, dtype=torch.int32, device=dev)
    L.check(L.lib().mn_setpts_t12(ctypes.byref(bins), P, L.ptr3(xs), int(bool(prec64)),
                                  L.ptr3(_rows(i1, dim)), L.ptr3(_rows(fr, dim)), L.ptr(key),
                                  L.stream()), "setpts")
    return i1, fr, key


def sort_keys(key, nbits):
    """Stable argsort of uint32 keys (stored in int32 tensors): (sorted, perm)."""
    skey, perm, _ = sort_pairs(key, nbits, [])
    return skey, perm


def sort_pairs(key, nbits, cols, outs=None, skey=None, perm=None, ws=None):
    """Stable sort of uint32 keys on their low nbits bits, carrying 32-bit
    payload columns (int32/float32 tensors of P elements) into outs:
    (sorted keys, perm, sorted columns). Outputs and the workspace are new
    tensors unless given."""
    P = key.numel()
    lib = L.lib()
    ncols = len(cols)
    ws_bytes = int(lib.mn_sort_pairs_workspace_bytes(P, ncols))
    if ws is None or ws.numel() < ws_bytes:
        ws = torch.empty(ws_bytes, dtype=torch.uint8, device=key.device)
    skey = torch.empty_like(key) if skey is None else skey
    perm = torch.empty_like(key) if perm is None else perm
    if outs is None:
        outs = [torch.empty_like(c) for c in cols]
    cin = (ctypes.c_void_p * max(1, ncols))(*[c.data_ptr() for c in cols])
    cout = (ctypes.c_void_p * max(1, ncols))(*[c.data_ptr() for c in outs])
    L.check(lib.mn_sort_pairs(P, int(nbits), L.ptr(key), L.ptr(skey), L.ptr(perm), ncols, cin,
                              cout, L.ptr(ws), ws.numel(), L.stream()), "sort")
    return skey, perm, outs


def gather_points(perm, i1, fr, extra=None):
    dim, P = i1.shape
    i1s = torch.empty_like(i1)
    frs = torch.empty_like(fr)
    ext = torch.empty_like(extra) if extra is not None else None
    L.check(L.lib().mn_gather_points(dim, P, L.ptr(perm), L.ptr3(_rows(i1, dim)),
                                     L.ptr3(_rows(fr, dim)), L.ptr3(_rows(i1s, dim)),
                                     L.ptr3(_rows(frs, dim)), L.ptr(extra), L.ptr(ext),
                                     L.stream()), "gather_points")
    return i1s, frs, ext


def build_subproblems(bins, skey, msub=MSUB):
    """(info[nsub, 3] = (bin, start, count), nsub). Blocks on one 8-byte read."""
    P = skey.numel()
    lib = L.lib()
    max_sub = bins.nbins + P // msub + 1
    info = torch.empty((max_sub, 3), dtype=torch.int32, device=skey.device)
    ws = torch.empty(int(lib.mn_subproblem_workspace_bytes(ctypes.byref(bins))),
                     dtype=torch.uint8, device=skey.device)
    nsub = ctypes.c_int64(0)
    L.check(lib.mn_build_subproblems(ctypes.byref(bins), P, L.ptr(skey), int(msub), L.ptr(info),
                                     max_sub, ctypes.byref(nsub), L.ptr(ws), ws.numel(),
                                     L.stream()), "subproblems")
    return info, int(nsub.value)


ZSTREAM_M = (16, 16, 8)  # bins of the streaming 3D interpolation


def zstream_eligible(dim, w):
    """True when the streaming 3D interpolation is selected (MN_INTERP=zstream,
    3D, 2 <= w <= 12). It reads the grid 1.7x instead of 4.3x, but measured
    slower than 8^3 tiles at 2e7 points / 512^3 (2.2 vs 2.0 ms: its window
    slides are not cache-line aligned and random gathers conflict in LDS),
    so the tiles are the default."""
    if os.environ.get("MN_INTERP", "") != "zstream":
        return False
    return dim == 3 and 2 <= w <= 12


class SortedPoints:
    """Bin-sorted point state of one point set on one fine grid: sorted cells
    and fractions, perm, and either the subproblem table (tiles) or the
    start of every bin (kind "zstream", bins of ZSTREAM_M)."""

    def __init__(self, bins, i1, fr, key, extra=None, msub=MSUB, stream=False):
        self.kind = "zstream" if stream else "tiles"
        self.bins = bins
        self.P = i1.shape[1]
        dim = bins.dim
        self.i1s = torch.empty_like(i1)
        self.frs = torch.empty_like(fr)
        cols = _rows(i1, dim) + _rows(fr, dim)
        outs = _rows(self.i1s, dim) + _rows(self.frs, dim)
        if extra is not None:
            cols += [extra.real.contiguous(), extra.imag.contiguous()]
            outs += [torch.empty_like(cols[-2]), torch.empty_like(cols[-1])]
        skey, self.perm, out = sort_pairs(key, key_bits(bins), cols, outs)
        self.extra = torch.complex(out[2 * dim], out[2 * dim + 1]) if extra is not None else None
        del out, outs, cols
        if stream:
            self.bstart = torch.empty(bins.nbins + 1, dtype=torch.int32, device=key.device)
            L.check(L.lib().mn_bin_starts(ctypes.byref(bins), self.P, L.ptr(skey),
                                          L.ptr(self.bstart), L.stream()), "bin starts")
            self.info, self.nsub = None, 0
        else:
            self.bstart = None
            self.info, self.nsub = build_subproblems(bins, skey, msub)
        self.skey = skey

    def i1_rows(self):
        return _rows(self.i1s, self.bins.dim)

    def fr_rows(self):
        return _rows(self.frs, self.bins.dim)


def fill_zero(t):
    L.check(L.lib().mn_fill_zero(L.ptr(t), t.numel() * t.element_size(), L.stream()),
            "fill_zero")


def zsweep_eligible(dim, w, n_up):
    """True when the owner-computes z-sweep spread applies: 3D, w <= 8, the
    x and y fine-grid sizes multiples of 8 (>= 16) and at most 2^23 sort keys
    ((n0/8)(n1/8) ceil(n2/8) 16, e.g. 512^3 or 1024^2 x 256). MN_SPREAD=tiles
    forces the LDS-tile spread instead."""
    if os.environ.get("MN_SPREAD", "") == "tiles":
        return False
    if dim != 3 or w > 8 or not all(n % 8 == 0 and n >= 16 for n in n_up[:2]) or n_up[2] < 8:
        return False
    return (n_up[0] // 8) * (n_up[1] // 8) * (-(-n_up[2] // 8)) * 16 <= 1 << 23


def zsweep_segment(n):
    """z-segment (cells) per wavefront of a sweep over the grid or extents n:
    the one that minimises rounds x (zseg + 8), a wave sweeping its segment and
    the chunk below it and about 2048 waves running at once. Measured, us, spread / z-gather, the chosen length
    and 256 cells: 5e5 points on 128^3, w = 6 (16) 72 / 40 and 206 / 157, 2e6 on
    256^3 (128) 168 / 149 and 232 / 251, 3e6 on 384 x 400 x 432, w = 7 (64)
    423 / 668 and 465 / 740; 512^3 keeps 256."""
    blocks = (n[0] // 8) * (n[1] // 8)

    def cost(z):
        return max(1.0, blocks * (-(-n[2] // z)) / 2048.0) * (min(z, n[2]) + 8)

    return min((256, 128, 64, 32, 16, 8), key=cost)


def zsweep_extents(dim, w, n_up):
    """Extents that let the z-sweep (and the z-gather) serve a 3D grid off its
    blocks: every axis holds the grid and the w - 1 cells footprints reach past
    it, rounded up to whole blocks and chunks, and the transform folds (or
    fills) that overhang. None where it does not apply: the sweep's own limits,
    a transform that cannot take extents, grids the sweep takes as they are."""
    if dim != 3 or zsweep_eligible(dim, w, n_up) or w > 8 or min(n_up) < 16:
        return None
    if not fftg_supported(n_up) or n_up[2] > 2048:
        return None
    ext = [-(-(int(n) + w - 1) // 8) * 8 for n in n_up]
    return ext if zsweep_eligible(dim, w, ext) else None


def tiles_beat_extents(w, n_up, ext, P):
    """True when dense points on a small grid stored with extents are better
    spread by tiles, up to w = 4: there a wave owns one 8-cell chunk and sweeps
    the one below as well. Measured, us, sweep / tiles: 50 x 160 x 72, w = 2, 0.3
    points a cell 54 / 46, 0.7 76 / 52; w = 4, 0.3 66 / 78, 0.7 104 / 88, 3.0
    302 / 228; 90 x 100 x 120, w = 2, 0.7 107 / 82, 6.0 531 / 388; w = 4, 0.7
    148 / 148, 6.0 870 / 624; w = 5 1085 / 1160; 72 x 90 x 288 (two chunks),
    w = 4, 1.4 290 / 316."""
    return (w <= 4 and zsweep_segment(ext) == 8
            and P > 0.6 * float(n_up[0]) * float(n_up[1]) * float(n_up[2]))


def sweep_load(pts):
    """Device int32: the points visited by the most loaded wave of a sweep."""
    load = torch.empty(1, dtype=torch.int32, device=pts.dev)
    if pts.kind == "ymfma":
        yseg = ymfma_segment([int(pts.bins.n[0]), int(pts.bins.n[1])])
        L.check(L.lib().mn_ymfma_maxload(ctypes.byref(pts.bins), yseg, L.ptr(pts.ystart),
                                         L.ptr(load), L.stream()), "ymfma load")
    else:
        L.check(L.lib().mn_zsweep_maxload(ctypes.byref(pts.bins), int(pts.kind == "zgather"),
                                          pts.zseg, L.ptr(pts.zstart), L.ptr(load), L.stream()),
                "zsweep load")
    return load


# points a us of one sweep wave, and us the tile kernels, which split crowded
# bins, take for 1000 points per unit of w. On radial points a y-window wave does
# 51 to 53; the 3D ones 25 to 28 and 14 to 18, put lower here: so the tiles were
# faster, or 5 us slower at most, in every set handed over (3e4 to 5e6 points).
_SWEEP_RATES = {"zsweep": (20.0, 0.04), "zgather": (8.0, 0.017), "ymfma": (52.0, 0.012)}


def sweep_balanced(load, kind, w, P, slack=1.0, repoint=False):
    """Whether a sweep is not held up by crowded points: its time is at least
    that of its most loaded wave (load points), which should not exceed slack
    times what the tile kernels take for all points. A step that re-points a
    plan also pays for the tiles' own point state after the sweep's (us, set
    and transform with the tiles / the sweep, radial points: 2D, w = 7, 1e6 on
    2048^2 472 / 387, 3e5 398 / 218; 3D, w = 2, 3e4 on 90 x 100 x 120
    310 / 203): 165 us and 30 for every 1e6 points more."""
    per_us, tile_us = _SWEEP_RATES[kind]
    setup = 165.0 + 30e-6 * P if repoint else 0.0
    return load / per_us <= slack * (30.0 + tile_us * 1e-3 * w * P) + setup


def sweep_sums_short(load, w, zseg):
    """Whether fp32 sums of the most loaded wave (load points) stay as near to
    64 bits as the tiles' fp64 sums of fp32 weights were. They add 1.6e-7 times
    the root of the points per cell: none of the error up to w = 5, as much as
    the tiles had at 20 points a cell for w = 6 (1.164e-5 both) and past 8 for
    wider kernels. Relative errors at 0.3 / 3 / 8 / 20 points per cell, 90 x 100
    x 120, against those tiles: w = 8 2.9e-7 / 3.9e-7 / 5.3e-7 / 7.7e-7 and
    6.9e-7 to 7.0e-7, w = 7 1.32e-6 / 1.35e-6 / 1.38e-6 / 1.45e-6 and 1.45e-6.
    The bound is the load of so many points spread evenly."""
    if w <= 5:
        return True
    per_cell = 20.0 if w == 6 else 8.0
    return load <= per_cell * 64.0 * (zseg + 8) * ((8 + w - 1) / 8.0) ** 2


class ZSweepPoints:
    """Point state for the z-sweep spread (gather=False, kind "zsweep") or
    the z-gather interpolation (gather=True, kind "zgather"): packed point
    words and fractions (setpts), stably sorted together by the z-sweep key
    (points of a block and z-chunk grouped by class for the spread, ordered
    by the x cell of their first tap for the gather), and the key start
    table. Given the previous point set of the same plan (prev) with the
    same P and geometry, its device buffers are reused, so re-pointing
    allocates nothing; prev's contents are overwritten in stream order.
    ngrid: the periodic grid when bins describe larger extents (then ext is
    True and every footprint lies inside them). stable: the gather evaluates
    its weights without cancellation (always on extents)."""

    def __init__(self, bins, x64, prec64, prev=None, gather=False, ngrid=None, stable=False):
        lib = L.lib()
        dev = x64[0].device
        self.kind = "zgather" if gather else "zsweep"
        self.bins = bins
        self.P = P = x64[0].numel()
        self.K = K = int(lib.mn_zsweep_nkeys(ctypes.byref(bins)))
        same = (prev is not None and prev.P == P and prev.K == K and prev.dev == dev)
        self.dev = dev
        self._bufs = bufs = prev._bufs if same else {}

        def buf(name, shape, dtype):
            if name not in bufs:
                bufs[name] = torch.empty(shape, dtype=dtype, device=dev)
            return bufs[name]

        word = buf("word_in", P, torch.int32)
        fr = buf("fr_in", (3, P), torch.float32)
        self.ext = ngrid is not None
        self.stable = stable
        self.zseg = zsweep_segment([int(bins.n[d]) for d in range(3)])
        L.check(lib.mn_zsweep_setpts_ext(ctypes.byref(bins), L.i64x3(ngrid), int(gather), P,
                                         L.ptr3(x64), int(bool(prec64)), L.ptr(word),
                                         L.ptr3(_rows(fr, 3)), L.stream())
                if self.ext else
                (lib.mn_zgather_setpts if gather else lib.mn_zsweep_setpts)(
                    ctypes.byref(bins), P, L.ptr3(x64), int(bool(prec64)), L.ptr(word),
                    L.ptr3(_rows(fr, 3)), L.stream()), f"{self.kind} setpts")
        self.frs = buf("frs", (3, P), torch.float32)
        ws_bytes = int(lib.mn_sort_pairs_workspace_bytes(P, 3))
        self.word, self.perm, _ = sort_pairs(
            word, max(1, (K - 1).bit_length()), _rows(fr, 3), _rows(self.frs, 3),
            skey=buf("word", P, torch.int32), perm=buf("perm", P, torch.int32),
            ws=buf("ws", ws_bytes, torch.uint8))
        self.zstart = buf("zstart", K + 1, torch.int32)
        L.check(lib.mn_zsweep_starts(ctypes.byref(bins), P, L.ptr(self.word), L.ptr(self.zstart),
                                     L.stream()), "zsweep starts")

    def fr_rows(self):
        return _rows(self.frs, 3)


def ysweep_eligible(dim, w, n_up):
    """True when the owner-computes y-sweep spread applies: 2D, w <= 8, the x
    fine-grid size a multiple of 64 (>= 128) and at most 2^26 sort keys
    ((n0/64)*n1*2). MN_SPREAD=tiles forces the LDS-tile spread instead."""
    if os.environ.get("MN_SPREAD", "") == "tiles":
        return False
    return (dim == 2 and 2 <= w <= 8 and n_up[0] % 64 == 0 and n_up[0] >= 128
            and n_up[1] >= w and (n_up[0] // 64) * n_up[1] * 2 <= 1 << 26)


def ymfma_eligible(dim, w, n_up):
    """True when the 2D spread on the matrix cores (y-window MFMA sweep)
    applies: 2D, w <= 8, n0 a multiple of 16 (>= 32), n1 a multiple of 8
    (>= 16) and at most 2^25 sort keys ((n0/16)*(n1/8)*2). MN_SPREAD=tiles
    forces the LDS-tile spread, MN_SPREAD=ysweep the VALU y-sweep."""
    if os.environ.get("MN_SPREAD", "") in ("tiles", "ysweep"):
        return False
    return (dim == 2 and 2 <= w <= 8 and n_up[0] % 16 == 0 and n_up[0] >= 32
            and n_up[1] % 8 == 0 and 16 <= n_up[1] < 1 << 24
            and (n_up[0] // 16) * (n_up[1] // 8) * 2 <= 1 << 25)


class YSweepPoints:
    """Point state for the 2D y-sweep spread (mfma=False, kind "ysweep") or
    the y-window MFMA sweep (mfma=True, kind "ymfma"): packed point words and
    fractions, stably sorted together by the sweep's key, and the key start
    table. Buffers of the previous point set of the same plan (prev, same
    kind, P and geometry) are reused, as in ZSweepPoints."""

    def __init__(self, bins, x64, prec64, prev=None, mfma=False):
        lib = L.lib()
        dev = x64[0].device
        self.kind = "ymfma" if mfma else "ysweep"
        nkeys, setpts, starts = ((lib.mn_ymfma_nkeys, lib.mn_ymfma_setpts, lib.mn_ymfma_starts)
                                 if mfma else
                                 (lib.mn_ysweep_nkeys, lib.mn_ysweep_setpts, lib.mn_ysweep_starts))
        self.bins = bins
        self.P = P = x64[0].numel()
        self.K = K = int(nkeys(ctypes.byref(bins)))
        same = (prev is not None and prev.kind == self.kind and prev.P == P and prev.K == K
                and prev.dev == dev)
        self.dev = dev
        self._bufs = bufs = prev._bufs if same else {}

        def buf(name, shape, dtype):
            if name not in bufs:
                bufs[name] = torch.empty(shape, dtype=dtype, device=dev)
            return bufs[name]

        V2 = ctypes.c_void_p * 2
        word = buf("word_in", P, torch.int32)
        fr = buf("fr_in", (2, P), torch.float32)
        L.check(setpts(ctypes.byref(bins), P, V2(x64[0].data_ptr(), x64[1].data_ptr()),
                       int(bool(prec64)), L.ptr(word), V2(fr[0].data_ptr(), fr[1].data_ptr()),
                       L.stream()), f"{self.kind} setpts")
        self.frs = buf("frs", (2, P), torch.float32)
        ws_bytes = int(lib.mn_sort_pairs_workspace_bytes(P, 2))
        self.word, self.perm, _ = sort_pairs(
            word, max(1, (K - 1).bit_length()), _rows(fr, 2), _rows(self.frs, 2),
            skey=buf("word", P, torch.int32), perm=buf("perm", P, torch.int32),
            ws=buf("ws", ws_bytes, torch.uint8))
        self.ystart = buf("ystart", K + 1, torch.int32)
        L.check(starts(ctypes.byref(bins), P, L.ptr(self.word), L.ptr(self.ystart), L.stream()),
                f"{self.kind} starts")

    def fr_rows(self):
        return _rows(self.frs, 2)


class _Subset:
    """Points [s, e) of a group-sorted copy of a point state: the attributes
    the spread entry points read, as views of the copy's columns (frs and
    i1s are lists of per-dimension rows)."""

    def __init__(self, kind, bins, P, **views):
        self.kind = kind
        self.bins = bins
        self.P = P
        self.__dict__.update(views)

    def fr_rows(self):
        return list(self.frs)

    def i1_rows(self):
        return list(self.i1s)


class GroupSplit:
    """A point state partitioned by group label, for spreads of disjoint
    point subsets that visit every point once in total.

    glabel: int64 labels in caller order; labels outside [0, G) are left
    out. One stable sort by label (carrying the spread's sorted columns)
    keeps each group's points in the state's key order, so each group is a
    contiguous, still key-sorted range. Iterating yields (g, subset) for the
    non-empty groups and builds the subset's start table just before it is
    used: z-/y-sweep key starts in one shared buffer (rebuilt in stream
    order, after the previous group's spread has read it), or the tile
    spread's subproblem table (sigma: spread_msub)."""

    def __init__(self, pts, glabel, G, sigma=2.0):
        self.pts = pts
        self.sigma = sigma
        self.G = G
        dim = pts.bins.dim
        gs = glabel[pts.perm.long()]
        gkey = torch.where((gs < 0) | (gs >= G), G, gs).to(torch.int32)
        del gs
        if pts.kind in ("zsweep", "ysweep", "ymfma"):
            cols = [pts.word, pts.perm] + _rows(pts.frs, dim)
        elif pts.kind == "tiles":
            cols = [pts.skey, pts.perm] + _rows(pts.frs, dim) + _rows(pts.i1s, dim)
        else:
            raise ValueError(f"no disjoint spread for point state {pts.kind!r}")
        skey, _, self.cols = sort_pairs(gkey, max(1, int(G).bit_length()), cols)
        del gkey
        bounds = torch.arange(G + 1, dtype=torch.int32, device=skey.device)
        self.starts = torch.searchsorted(skey, bounds).cpu().tolist()
        self._startbuf = None

    def __iter__(self):
        pts, dim, lib, c = self.pts, self.pts.bins.dim, L.lib(), self.cols
        for g in range(self.G):
            s, e = self.starts[g], self.starts[g + 1]
            if e == s:
                continue
            frs = [r[s:e] for r in c[2:2 + dim]]
            if pts.kind == "tiles":
                sub = _Subset("tiles", pts.bins, e - s, perm=c[1][s:e], skey=c[0][s:e], frs=frs,
                              i1s=[r[s:e] for r in c[2 + dim:2 + 2 * dim]])
                sub.info, sub.nsub = build_subproblems(
                    pts.bins, sub.skey, spread_msub(pts.bins, sub.P, self.sigma))
                yield g, sub
                continue
            if self._startbuf is None:
                self._startbuf = torch.empty(pts.K + 1, dtype=torch.int32,
                                             device=pts.perm.device)
            sub = _Subset(pts.kind, pts.bins, e - s, perm=c[1][s:e], word=c[0][s:e], frs=frs,
                          K=pts.K, ext=getattr(pts, "ext", False), zseg=getattr(pts, "zseg", 0))
            starts_fn = {"zsweep": lib.mn_zsweep_starts, "ysweep": lib.mn_ysweep_starts,
                         "ymfma": lib.mn_ymfma_starts}[pts.kind]
            L.check(starts_fn(ctypes.byref(pts.bins), sub.P, L.ptr(sub.word),
                              L.ptr(self._startbuf), L.stream()), f"{pts.kind} starts")
            if pts.kind == "zsweep":
                sub.zstart = self._startbuf
            else:
                sub.ystart = self._startbuf
            yield g, sub


def ysweep_vectors_per_wave(B):
    """Vectors one y-sweep wavefront carries (the kernel's rule): the
    largest of 8, 4, 2, 1 not above B."""
    return 8 if B >= 8 else 4 if B >= 4 else 2 if B >= 2 else 1


def ysweep_segment(n_up, B):
    """y-segment per wavefront: the longest power of two (<= 256) that still
    gives at least 8192 / VB wavefronts (VB vectors per wavefront), but at
    least 32 (each segment re-reads the w - 1 rows below it to warm its
    window). Measured at 2048^2, 1e7 points, w = 7: 32 for B = 1 (0.49 ms;
    0.58 at 16, 0.84 at 64); 64 for B = 8, VB = 8 (2.19 ms; 2.39 at 32)."""
    vb = ysweep_vectors_per_wave(B)
    groups = -(-B // vb)
    nbx = n_up[0] // 64
    yseg = 256
    while yseg > 32 and nbx * (-(-n_up[1] // yseg)) * groups * vb < 8192:
        yseg //= 2
    return yseg


def spread_ysweep(pts, beta, cs, grids):
    """grids[b] = spread(cs[b]) for B vectors (cs: (B, P) or (P,), caller
    order) with the 2D y-sweep; grids are fully overwritten."""
    B = 1 if cs.dim() == 1 else int(cs.shape[0])
    n_up = [int(pts.bins.n[0]), int(pts.bins.n[1])]
    V2 = ctypes.c_void_p * 2
    L.check(L.lib().mn_spread_ysweep(ctypes.byref(pts.bins), float(beta), pts.P, B,
                                     ysweep_segment(n_up, B), L.ptr(pts.ystart), L.ptr(pts.perm),
                                     L.ptr(pts.word), V2(pts.frs[0].data_ptr(), pts.frs[1].data_ptr()),
                                     L.ptr(cs), L.ptr(grids), L.stream()), "spread_ysweep")


def tiles_beat_ysweep(bins, w, P):
    """True when many points on a grid only the VALU y-sweep fits are better
    spread by the matrix-core tiles (bins: the tiles'): w = 7, us, sweep /
    tiles, 2e5 points on 256 x 270 412 / 34, 1e6 on 1024 x 900 194 / 63
    (radial 2366 / 89), 1e7 on 2048 x 2250 486 / 325. MN_SPREAD=ysweep keeps
    the sweep."""
    return (os.environ.get("MN_SPREAD", "") != "ysweep" and P >= 1 << 17
            and bins.m[0] + w - 1 <= 16)


def ymfma_segment(n_up):
    """y-segment per wavefront of the y-window MFMA sweep: the one (8 to 256
    cells) that minimises rounds x (yseg + 8), as zsweep_segment, for one wave
    per block (up to 8 vectors), so that a batch sums as its vectors do alone.
    Measured, us, w = 7, one vector / 8, at the chosen length and at 32 cells:
    1e5 points on 256^2 (8) 19 / 57 and 34 / 108; 1e6 on 512^2 (8) 51 / 178 and
    72 / 250; 1e7 on 2048^2 (128) 265 / 940 and 324 / 1036 (327 / 974 at 64).
    Sets that crowd like longer segments less: 1e7 radial points there 16 %
    slower than at 64."""
    blocks = n_up[0] // 16

    def cost(y):
        return max(1.0, blocks * (-(-n_up[1] // y)) / 2048.0) * (min(y, n_up[1]) + 8)

    return min((256, 128, 64, 32, 16, 8), key=cost)


def spread_ymfma(pts, beta, cs, grids):
    """grids[b] = spread(cs[b]) for B vectors (cs: (B, P) or (P,), caller
    order) with the y-window MFMA sweep; grids are fully overwritten. Several
    vectors are first transposed to point-major (P, B), so that a point
    visit gathers its strengths in one run rather than one sector per
    vector."""
    B = 1 if cs.dim() == 1 else int(cs.shape[0])
    n_up = [int(pts.bins.n[0]), int(pts.bins.n[1])]
    V2 = ctypes.c_void_p * 2
    pm = 0
    if B > 1:
        _require(cs.is_contiguous() and cs.dtype == torch.complex64,
                 "spread_ymfma: cs must be a contiguous complex64 (B, P) tensor")
        ct = torch.empty((int(cs.shape[1]), B), dtype=torch.complex64, device=cs.device)
        L.check(L.lib().mn_pointmajor_c64(B, int(cs.shape[1]), L.ptr(cs), L.ptr(ct), L.stream()),
                "pointmajor")
        cs = ct
        pm = 1
    L.check(L.lib().mn_spread_ymfma(ctypes.byref(pts.bins), float(beta), pts.P, B,
                                    ymfma_segment(n_up), L.ptr(pts.ystart), L.ptr(pts.perm),
                                    L.ptr(pts.word), V2(pts.frs[0].data_ptr(), pts.frs[1].data_ptr()),
                                    L.ptr(cs), pm, L.ptr(grids), L.stream()), "spread_ymfma")


def permute_c64(perm, c, out):
    """out[j] = c[perm[j]] (complex64 strengths into sorted order)."""
    L.check(L.lib().mn_permute_c64(perm.numel(), L.ptr(perm), L.ptr(c), L.ptr(out), L.stream()),
            "permute")


def spread_zsweep(pts, beta, c, grid, pre=None, zseg=None, presorted=False):
    """grid = spread(c) with the owner-computes z-sweep (overwrites grid).
    c is in caller order, or in sorted order when presorted."""
    if pts.ext:  # (c may hold more points than a subset pts indexes)
        _require(pre is None, "spread_zsweep: no prephase on a grid stored with extents")
        L.check(L.lib().mn_spread_zsweep_ext(
            ctypes.byref(pts.bins), float(beta), pts.P, 1, int(zseg or pts.zseg),
            L.ptr(pts.zstart), None if presorted else L.ptr(pts.perm), L.ptr(pts.word),
            L.ptr3(pts.fr_rows()), L.ptr(c), L.ptr(grid), L.stream()), "spread_zsweep")
        return
    L.check(L.lib().mn_spread_zsweep(ctypes.byref(pts.bins), float(beta), pts.P,
                                     int(zseg or pts.zseg),
                                     L.ptr(pts.zstart), None if presorted else L.ptr(pts.perm),
                                     L.ptr(pts.word), L.ptr3(pts.fr_rows()), L.ptr(c), L.ptr(pre),
                                     L.ptr(grid), L.stream()), "spread_zsweep")


def spread_zsweep_batch(pts, beta, cs, grids, zseg=None, presorted=False):
    """grids[b] = spread(cs[b]) for B vectors with the z-sweep, one launch
    with a wave per (block, vector) (overwrites grids)."""
    B = cs.shape[0]
    _require(grids.shape[0] == B and cs.shape[1] == pts.P and cs.is_contiguous()
             and grids.is_contiguous(), "spread_zsweep_batch: cs must be (B, P) and grids "
             "(B, n0, n1, n2), both contiguous")
    fn = L.lib().mn_spread_zsweep_ext if pts.ext else L.lib().mn_spread_zsweep_batch
    L.check(fn(ctypes.byref(pts.bins), float(beta), pts.P, B, int(zseg or pts.zseg),
               L.ptr(pts.zstart), None if presorted else L.ptr(pts.perm), L.ptr(pts.word),
               L.ptr3(pts.fr_rows()), L.ptr(cs), L.ptr(grids), L.stream()), "spread_zsweep_batch")


def spread(pts, beta, c, grid, pre=None, accumulate=False):
    """grid = spread(c) (or grid += spread(c) with accumulate=True)."""
    fn = L.lib().mn_spread_accumulate if accumulate else L.lib().mn_spread
    L.check(fn(ctypes.byref(pts.bins), float(beta), pts.P, pts.nsub, L.ptr(pts.info),
               L.ptr(pts.perm), L.ptr3(pts.i1_rows()), L.ptr3(pts.fr_rows()), L.ptr(c),
               L.ptr(pre), L.ptr(grid), L.stream()), "spread")


def spread_c128(pts, beta, c, grid128, pre=None):
    """grid128 (complex128) = spread(c) with fp64 products and accumulation."""
    L.check(L.lib().mn_spread_c128(ctypes.byref(pts.bins), float(beta), pts.P, pts.nsub,
                                   L.ptr(pts.info), L.ptr(pts.perm), L.ptr3(pts.i1_rows()),
                                   L.ptr3(pts.fr_rows()), L.ptr(c), L.ptr(pre), L.ptr(grid128),
                                   L.stream()), "spread_c128")


def t3_tile_bins(w, n):
    """Bins of the type-3 LDS-tile spread. With w <= 16 the matrix-core
    kernel takes the tiles, so bins are 17 - w cells wide: padded tiles of 16
    cells per dim (one 16 x 16 MFMA tile per x plane). MN_T3_TILE_MFMA=0
    selects the LDS-atomic kernel and the LDS budget's bins instead."""
    if w <= 16 and os.environ.get("MN_T3_TILE_MFMA", "") != "0":
        return make_bins(3, w, n, m=[max(1, min(17 - w, int(k))) for k in n])
    return make_bins(3, w, n, cell_bytes=SPREAD_CELL_BYTES)


OWNER_M = 16   # owner-computes spread bins: 16^3 fp64 complex cells = 64 KB of LDS


def owner_bins(w, n):
    """Owner-computes spread bins: 16 cells per dim, except a last dim of at
    most 18 cells, which stays whole (one bin along it: no split columns and
    no second z-owner per point; 16*16*18 cells still fit two workgroups per
    CU)."""
    m = [min(OWNER_M, k) for k in n]
    if n[2] <= 18:
        m[2] = n[2]
    return make_bins(3, w, n, m=m)


def spread_owner_c128(pts, beta, c, grid128, pre=None):
    """Owner-computes 3D spread into a complex128 grid that it fully
    overwrites (no zero fill); pts must carry bin starts (kind "zstream")."""
    _require(pts.bstart is not None and grid128.dtype == torch.complex128
             and grid128.numel() >= int(np.prod([pts.bins.n[d] for d in range(3)])),
             "spread_owner_c128: needs a point state with bin starts and a complex128 grid of "
             "the fine-grid size")
    L.check(L.lib().mn_spread_owner_c128(ctypes.byref(pts.bins), float(beta), pts.P,
                                         L.ptr(pts.bstart), L.ptr(pts.perm), L.ptr3(pts.i1_rows()),
                                         L.ptr3(pts.fr_rows()), L.ptr(c),
                                         None if pre is None else L.ptr(pre), L.ptr(grid128),
                                         L.stream()), "spread_owner_c128")


def spread_batch(pts, beta, cs, grids):
    L.check(L.lib().mn_spread_batch(ctypes.byref(pts.bins), float(beta), pts.P, pts.nsub,
                                    L.ptr(pts.info), L.ptr(pts.perm), L.ptr3(pts.i1_rows()),
                                    L.ptr3(pts.fr_rows()), int(cs.shape[0]), L.ptr(cs),
                                    L.ptr(grids), L.stream()), "spread_batch")


def interp_direct(pts, beta, grid, out, post=None):
    """3D gather without staged tiles: one thread per sorted point reads its
    w^3 taps from the grid (sparse point sets)."""
    L.check(L.lib().mn_interp_direct(ctypes.byref(pts.bins), float(beta), pts.P, L.ptr(pts.perm),
                                     L.ptr3(pts.i1_rows()), L.ptr3(pts.fr_rows()), L.ptr(grid),
                                     L.ptr(post), L.ptr(out), L.stream()), "interp direct")


def interp_direct_preferred(pts, w, n_up):
    """True when the direct gather should beat the staged one: its w^3 taps
    per point against the staged path's padded tile per subproblem (or ~1.7
    reads of the grid for the z-streaming path). Measured on MI355X (taps /
    staged cells: staged ms, direct ms): 11.4: 0.43, 0.53 (1e6 targets on
    240^3); 2.3-2.6: 2.62, 2.20 and 6.43, 3.14 (4e6 targets on 640^3 and on
    5400^2 x 24); 0.6: 2.42, 0.74 and 4.17, 1.19 (1e6 targets on the same
    grids). The crossover lies between 2.6 and 11.4; 5 is used."""
    if pts.bins.dim != 3:
        return False
    direct = float(pts.P) * w ** 3
    if pts.kind == "zstream":
        staged = 1.7 * float(np.prod([float(n) for n in n_up]))
    else:
        staged = float(pts.nsub) * float(np.prod([pts.bins.m[d] + w - 1 for d in range(3)]))
    return direct < 5.0 * staged


def zgather_preferred(P, w, n_up, sigma=2.0):
    """True when the z-gather interpolation should beat the direct and the
    staged-tile gathers for P points on the 3D fine grid n_up. The direct
    gather reads P w^3 taps, the z-gather (8 + w - 1)^2 columns of 8 new
    z-cells for every 8x8-column block and z-chunk that holds points (16 after
    a skipped chunk), expected over uniform points. On grids within the
    last-level cache (2^25 cells) it has to halve the traffic several times
    over (a factor 5, as between the direct and the staged-tile gathers), on
    larger ones, where every halo cell comes from memory, far less; and up to
    w = 5 its matrix products, padded to 16 rows, cost as much as the tiles'
    taps. Measured, us, z-gather / tiles: 384 x 400 x 432, 2e6 points, w = 4
    341 / 266, w = 5 349 / 420, w = 8 439 / 866; 200 x 192 x 180, 1.4e6, w = 4
    93 / 67, w = 5 98 / 75, w = 6 104 / 104, w = 8 141 / 235; 1.1e7, w = 5
    555 / 672. (Below 2^18 points the w <= 5 difference is some us.) On grids
    stored with extents the tiles have all points up to w = 5 there: 1.7e6 on
    50 x 160 x 72, w = 5, 157 / 104, 5.9e6 on 90 x 100 x 120 412 / 241, 2.5e5 on
    54 x 50 x 72, w = 4, 73 / 39; 57600 on 50 x 160 x 72, w = 5, 38 / 40.
    Between the factors the other gathers read the grid in fp32, so there the
    z-gather's split operands need the weights that make up for them
    (zgather_stable), and below sigma = 2 they do not: 2e6 points on 360^3 at
    sigma = 1.25, w = 7, 1.5048e-4 from 64 bits against 1.5044e-4."""
    ratio = _zgather_ratio(P, w, n_up)
    cells = float(n_up[0]) * float(n_up[1]) * float(n_up[2])
    if cells >= 2.0 ** 25:
        return ratio >= (1.5 if sigma >= 2.0 else 5.0)
    if w <= 5 and (n_up[0] % 8 or n_up[1] % 8):
        return False
    if w <= 5 and P >= 1 << 18 and (w < 5 or P < 1.2 * cells):
        return False
    return ratio >= 5.0


def _zgather_ratio(P, w, n_up):
    """Taps of the direct gather over the cells the z-gather reads."""
    nchunks = (n_up[0] / 8.0) * (n_up[1] / 8.0) * -(-n_up[2] // 8)
    lam = float(P) / nchunks
    busy = nchunks * -np.expm1(-lam)
    return float(P) * w ** 3 / ((8 + w - 1) ** 2 * 8.0 * busy * (1.0 + np.exp(-lam)))


def zgather_stable(P, w, n_up):
    """Whether a z-gather on its own grid evaluates the kernel's exponent
    without cancellation: where it takes points from the fp32 gathers (below
    the factor 5 of zgather_preferred) it must be no further from 64 bits
    than they are. 3e6 points on 384^3, z-gather / with this exponent / fp32
    gather: w = 6 1.1950e-5 / 1.1933e-5 / 1.1944e-5, w = 7 1.620e-6 / 1.438e-6
    / 1.578e-6, w = 8 8.64e-7 / 3.43e-7 / 7.89e-7; the times are equal
    (787 and 780 us at w = 7)."""
    return _zgather_ratio(P, w, n_up) < 5.0


def interp_zgather(pts, beta, grids, outs, B=1, zseg=None):
    """3D interpolation over the z-sweep point state: B grids (B x n_up)
    into B output vectors of P values in caller order (outs: B x P)."""
    stable = pts.ext or pts.stable
    fn = L.lib().mn_interp_zgather_ext if stable else L.lib().mn_interp_zgather
    L.check(fn(ctypes.byref(pts.bins), float(beta), pts.P, int(B), int(zseg or pts.zseg),
               L.ptr(pts.zstart), L.ptr(pts.perm), L.ptr(pts.word), L.ptr3(pts.fr_rows()),
               L.ptr(grids), L.ptr(outs), L.stream()), "interp_zgather")


def interp(pts, beta, grid, out, post=None):
    if pts.kind == "zstream":
        L.check(L.lib().mn_interp_zstream(ctypes.byref(pts.bins), float(beta), pts.P,
                                          L.ptr(pts.bstart), L.ptr(pts.perm),
                                          L.ptr3(pts.i1_rows()), L.ptr3(pts.fr_rows()),
                                          L.ptr(grid), L.ptr(post), L.ptr(out), L.stream()),
                "interp")
        return
    L.check(L.lib().mn_interp(ctypes.byref(pts.bins), float(beta), pts.P, pts.nsub,
                              L.ptr(pts.info), L.ptr(pts.perm), L.ptr3(pts.i1_rows()),
                              L.ptr3(pts.fr_rows()), L.ptr(grid), L.ptr(post), L.ptr(out),
                              L.stream()), "interp")


def kernel_dec(N, n_up, quad, device):
    """fp32 mode deconvolution factors per dim, 1 / phihat(2 pi k / n_up[d]);
    quad: the kernel's quadrature (nodes, weights)."""
    dq, fq = quad
    out = torch.empty(sum(N), dtype=torch.float32, device=device)
    L.check(L.lib().mn_kernel_dec(len(N), L.i64x3(N), L.i64x3(n_up), dq.ctypes.data,
                                  fq.ctypes.data, len(dq), L.ptr(out), L.stream()), "kernel_dec")
    return list(out.split([int(n) for n in N]))


def crop_deconv(n_up, N, grid, decs, fk, batch=1):
    dim = len(N)
    L.check(L.lib().mn_crop_deconv(dim, L.i64x3(n_up), L.i64x3(N), int(batch), L.ptr(grid),
                                   L.ptr3(decs), L.ptr(fk), L.stream()), "crop_deconv")


def pad_deconv(n_up, N, fk, decs, grid, batch=1):
    dim = len(N)
    L.check(L.lib().mn_pad_deconv(dim, L.i64x3(n_up), L.i64x3(N), int(batch), L.ptr(fk),
                                  L.ptr3(decs), L.ptr(grid), L.stream()), "pad_deconv")


def fftp_supported(n_up):
    """True when the pruned per-axis FFT applies (power-of-two fine grid
    sizes in [16, 4096]); MN_FFT=rocfft forces full rocFFT + crop/pad."""
    if os.environ.get("MN_FFT", "") == "rocfft":
        return False
    return bool(L.lib().mn_fftp_supported(len(n_up), L.i64x3(n_up)))


def fftp_work_bytes(n_up, N, batch=1):
    return int(L.lib().mn_fftp_work_bytes(len(N), L.i64x3(n_up), L.i64x3(N), int(batch)))


def fft_crop_deconv(n_up, N, grid, decs, fk, isign, work, batch=1):
    """fk = crop(FFT(grid)) * prod_d dec_d with the pruned per-axis FFT."""
    L.check(L.lib().mn_fft_crop_deconv(len(N), L.i64x3(n_up), L.i64x3(N), int(batch), int(isign),
                                       L.ptr(grid), L.ptr3(decs), L.ptr(work),
                                       0 if work is None else work.numel(), L.ptr(fk),
                                       L.stream()), "fft_crop_deconv")


def pad_deconv_fft(n_up, N, fk, decs, grid, isign, work, batch=1):
    """grid = FFT(pad(fk * prod_d dec_d)) with the pruned per-axis FFT."""
    L.check(L.lib().mn_pad_deconv_fft(len(N), L.i64x3(n_up), L.i64x3(N), int(batch), int(isign),
                                      L.ptr(fk), L.ptr3(decs), L.ptr(work),
                                      0 if work is None else work.numel(), L.ptr(grid),
                                      L.stream()), "pad_deconv_fft")


def fftg_supported(n_up):
    """True when the general pruned FFT applies (5-smooth fine-grid sizes);
    MN_FFT=rocfft forces full rocFFT + crop/pad."""
    if os.environ.get("MN_FFT", "") == "rocfft":
        return False
    return bool(L.lib().mn_fftg_supported(len(n_up), L.i64x3(n_up)))


def fftg_work_bytes(n_up, N, batch=1):
    return int(L.lib().mn_fftg_work_bytes(len(N), L.i64x3(n_up), L.i64x3(N), int(batch)))


def fftg_crop_deconv(n_up, N, grid, decs, fk, isign, work, batch=1, ext=None):
    """fk = crop(FFT(grid)) * prod_d dec_d with the general pruned FFT; the
    grid is stored with extents ext (n_up when None)."""
    L.check(L.lib().mn_fftg_crop_deconv(len(N), L.i64x3(n_up), L.i64x3(N),
                                        L.i64x3(n_up if ext is None else ext), int(batch),
                                        int(isign), L.ptr(grid), L.ptr3(decs), L.ptr(work),
                                        0 if work is None else work.numel(), L.ptr(fk),
                                        L.stream()), "fftg_crop_deconv")


def fftg_pad_deconv(n_up, N, fk, decs, grid, isign, work, batch=1, ext=None):
    """grid = FFT(pad(fk * prod_d dec_d)) with the general pruned FFT; the
    grid is stored with extents ext (n_up when None)."""
    L.check(L.lib().mn_fftg_pad_deconv(len(N), L.i64x3(n_up), L.i64x3(N),
                                       L.i64x3(n_up if ext is None else ext), int(batch),
                                       int(isign), L.ptr(fk), L.ptr3(decs), L.ptr(work),
                                       0 if work is None else work.numel(), L.ptr(grid),
                                       L.stream()), "fftg_pad_deconv")


def pad_deconv_c128(n_up, N, fk128, decs64, grid128, batch=1):
    """grid128 = pad(fk128 * prod_d dec_d), complex128 with fp64 factors."""
    L.check(L.lib().mn_pad_deconv_c128(len(N), L.i64x3(n_up), L.i64x3(N), int(batch), L.ptr(fk128),
                                       L.ptr3(decs64), L.ptr(grid128), L.stream()),
            "pad_deconv_c128")


def fft_f64(grid128, n_up, isign, batch=1):
    """In-place complex128 FFT (rocFFT double precision)."""
    L.check(L.lib().mn_fft_exec_f64(len(n_up), L.i64x3(n_up), int(batch), int(isign),
                                    L.ptr(grid128), L.stream()), "fft_f64")


def round_c64(src128, out64):
    L.check(L.lib().mn_round_c64(src128.numel(), L.ptr(src128), L.ptr(out64), L.stream()),
            "round_c64")


def fft64_lines_supported(n):
    return bool(L.lib().mn_fft64_lines_supported(int(n)))


FFT64_LAYOUTS = {"anb": 0, "lines_last": 1, "lines_first": 2}


def target_cells(n, w, R, margin=1):
    """[lo, hi) holding every tap of targets within R cells of the middle of an
    axis of n cells, the whole axis where they would wrap. The length is a
    multiple of 16 or 8 where that fits, so that strided line passes over the
    range have tiles of as many lines, and lo one of 8 where that is no longer."""
    lo = math.floor(0.5 * (n - w) - R) - margin
    hi = math.ceil(0.5 * (n + w) + R) + margin
    if lo < 0 or hi > n:
        return 0, n
    best = (0, n)
    for start in (lo - lo % 8, lo):
        for step in (16, 8):
            end = start + -(-(hi - start) // step) * step
            if end <= n and end - start < best[1] - best[0]:
                best = (start, end)
                break
    return best


def fft64_lines(A, nin, B, n, isign, src128, dec64, out, layout="anb", keep=None, rows=None):
    """One axis pass of the zero-padding fp64 line FFT: src128 (A, nin, B)
    complex128 -> out (A, n, B) ("anb"), (n, A*B) with the line index fastest
    ("lines_last") or (A*B, n) with each line contiguous ("lines_first"),
    complex128 or complex64 (by out's dtype). keep = (r0, r1) stores those
    outputs of each line only; rows = (period, (q0, q1), (c0, c1)) transforms
    the lines q * period + c in these ranges only (index a * B + b)."""
    _require(layout in FFT64_LAYOUTS, f"fft64_lines: layout must be one of {tuple(FFT64_LAYOUTS)}")
    c64 = out.dtype == torch.complex64
    _require(src128.dtype == torch.complex128 and src128.numel() >= A * nin * B,
             f"fft64_lines: src must be complex128 with at least {A * nin * B} elements")
    _require(out.numel() >= A * n * B and (c64 or out.dtype == torch.complex128),
             f"fft64_lines: out must be complex64/128 with at least {A * n * B} elements")
    _require(dec64 is None or (dec64.dtype == torch.float64 and dec64.numel() >= nin),
             f"fft64_lines: dec must be float64 with at least {nin} elements")
    part = None
    if keep is not None or rows is not None:
        period, q, c = rows or ((B, (0, A), (0, B)) if B > 1 else (A, (0, 1), (0, A)))
        part = (ctypes.c_int64 * 7)(*(keep or (0, n)), period, *q, *c)
    L.check(L.lib().mn_fft64_lines_part(int(A), int(nin), int(B), int(n), int(isign),
                                        L.ptr(src128), None if dec64 is None else L.ptr(dec64),
                                        L.ptr(out), int(c64), FFT64_LAYOUTS[layout], part,
                                        L.stream()), "fft64_lines")


def transpose_c128(Bt, R, C, src, out):
    """out[b][c][r] = src[b][r][c] for complex128 (Bt, R, C) -> (Bt, C, R)."""
    _require(src.dtype == torch.complex128 and out.dtype == torch.complex128,
             "transpose_c128: src and out must be complex128")
    _require(src.numel() >= Bt * R * C and out.numel() >= Bt * R * C,
             f"transpose_c128: src and out need at least {Bt * R * C} elements")
    L.check(L.lib().mn_transpose_c128(int(Bt), int(R), int(C), L.ptr(src), L.ptr(out),
                                      L.stream()), "transpose_c128")


def fft(grid, n_up, isign, batch=1):
    L.check(L.lib().mn_fft_exec(len(n_up), L.i64x3(n_up), int(batch), int(isign), L.ptr(grid),
                                L.stream()), "fft")


def expi(comps, isign, out):
    arr = (ctypes.c_void_p * len(comps))(*[c.data_ptr() for c in comps])
    L.check(L.lib().mn_expi(len(comps), arr, comps[0].numel(), int(isign), L.ptr(out),
                            L.stream()), "expi")


class StageTimer:
    """Optional per-stage HIP-event timing on the current stream."""

    def __init__(self, enabled):
        self.enabled = enabled
        self.events = []

    @contextlib.contextmanager
    def __call__(self, name):
        if not self.enabled:
            yield
            return
        a = torch.cuda.Event(enable_timing=True)
        b = torch.cuda.Event(enable_timing=True)
        a.record()
        yield
        b.record()
        self.events.append((name, a, b))

    def times_ms(self, sync=True):
        if sync:
            torch.cuda.synchronize()
        out = {}
        for name, a, b in self.events:
            out[name] = out.get(name, 0.0) + a.elapsed_time(b)
        return out
