"""The general pruned FFT (mn_fftg_*) against numpy on grids whose sizes are
not powers of two: every stage radix, axes split in two passes, tiles past the
last line, and grids stored with larger extents, whose overhang type 1 folds
in and type 2 fills."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _cplx(rng, shape):
    return (rng.standard_normal(shape) + 1j * rng.standard_normal(shape)).astype(np.complex64)


@pytest.mark.parametrize("n,ext", [
    ((4,), None), ((6,), None), ((10,), None), ((18,), None), ((90,), None), ((250,), None),
    ((320,), None), ((324,), None), ((486,), None), ((1024,), None), ((1080,), None),
    ((2000,), None), ((2048,), None), ((2160,), None), ((4374,), None), ((65536,), None),
    ((202500,), None),
    ((36, 50), None), ((36, 50), (48, 56)), ((30, 54), (44, 54)), ((2160, 6), None),
    ((6, 2250), None), ((20, 4500), None),
    ((12, 10, 18), None), ((18, 24, 30), (32, 32, 40)), ((18, 16, 30), (18, 16, 36)),
    ((20, 18, 16), (32, 18, 16)), ((4, 2160, 6), None),
])
@pytest.mark.parametrize("isign", [+1, -1])
def test_general_fft_vs_numpy(n, ext, isign, mn):
    from mlx_nufft_amd import _engine as E

    print(f"case fftg n={n} ext={ext} isign={isign}", flush=True)
    rng = np.random.default_rng(sum(n))
    dim, B = len(n), 3 if np.prod(n) < 1e4 else 1
    N = [max(1, (2 * k) // 3 - (k // 2) % 2) for k in n]
    ext = n if ext is None else ext
    assert E.fftg_supported(n)
    decs = [rng.uniform(0.5, 2.0, k).astype(np.float32) for k in N]
    dd = [torch.from_numpy(d).cuda() for d in decs]
    dec = decs[0].astype(np.float64)
    for d in decs[1:]:
        dec = np.multiply.outer(dec, d.astype(np.float64))
    work = torch.empty(max(1, E.fftg_work_bytes(n, N, B)), dtype=torch.uint8, device="cuda")
    axes = tuple(range(1, dim + 1))
    idx = np.ix_(range(B), *[np.arange(-(k // 2), k - k // 2) % m for k, m in zip(N, n)])
    # rounding: one ulp (2^-24) per butterfly level and input, twice over for
    # the twiddles, log2(prod n) levels at most
    tol = 2.0 ** -23 * np.log2(np.prod([float(k) for k in n]))

    def transform(G):
        if isign > 0:
            return np.fft.ifftn(G, axes=axes) * np.prod(n)
        return np.fft.fftn(G, axes=axes)

    grid = _cplx(rng, (B, *ext))
    fk = torch.full((B, *N), float("nan"), dtype=torch.complex64, device="cuda")
    E.fftg_crop_deconv(n, N, torch.from_numpy(grid).cuda(), dd, fk, isign, work, batch=B, ext=ext)
    G = grid.astype(np.complex128)
    for d in range(dim):  # the overhang folded back
        G = np.moveaxis(G, d + 1, 0)
        H = G[:n[d]].copy()
        H[:ext[d] - n[d]] += G[n[d]:]
        G = np.moveaxis(H, 0, d + 1)
    ref = transform(G)[idx] * dec
    assert np.linalg.norm(fk.cpu().numpy() - ref) <= tol * np.linalg.norm(ref)

    f2 = _cplx(rng, (B, *N))
    g2 = torch.full((B, *ext), float("nan"), dtype=torch.complex64, device="cuda")
    E.fftg_pad_deconv(n, N, torch.from_numpy(f2).cuda(), dd, g2, isign, work, batch=B, ext=ext)
    H = np.zeros((B, *n), np.complex128)
    H[idx] = f2 * dec
    R = transform(H)
    for d in range(dim):
        R = np.take(R, np.arange(ext[d]) % n[d], axis=d + 1)
    assert np.linalg.norm(g2.cpu().numpy() - R) <= tol * np.linalg.norm(R)


def test_general_fft_refusals(mn):
    from mlx_nufft_amd import _engine as E

    for n in ((14,), (4194306,), (2, 8), (22, 30)):
        assert not E.fftg_supported(n)
        assert E.fftg_work_bytes(n, n) == -1
    g = torch.zeros((12, 10), dtype=torch.complex64, device="cuda")
    dd = [torch.ones(4, device="cuda")] * 2
    fk = torch.zeros((4, 4), dtype=torch.complex64, device="cuda")
    work = torch.empty(E.fftg_work_bytes((12, 10), (4, 4)), dtype=torch.uint8, device="cuda")
    for ext in ((11, 10), (25, 10)):
        with pytest.raises(ValueError):
            E.fftg_crop_deconv((12, 10), (4, 4), g, dd, fk, 1, work, ext=ext)
    with pytest.raises(ValueError):
        E.fftg_crop_deconv((12, 10), (4, 4), g, dd, fk, 1, work[:8])
