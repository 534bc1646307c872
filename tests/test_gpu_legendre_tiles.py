"""The Legendre stage over its column tiles: one to five tiles of 32 columns per workgroup, tiles with columns past the last one, K ranges of one chunk and of
many, columns whose neighbours lie far above or below them and whose scale moves late in the sum, against float64."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# (nlat, nlon, lmax, mmax, rows): between them the launcher's five tile counts (few columns or few orders to a CU: one; 384 rows of many latitudes: four; rows of a
# whole state: five), one chunk of K and a last one of 1, 2, 15 and 16 rows, an odd and an even number of latitudes, orders past the last degree
CASES = [(3, 8, 2, 3, 1), (4, 8, 4, 5, 128), (33, 64, 33, 33, 8), (35, 64, 20, 33, 37), (61, 120, 61, 61, 33), (64, 128, 64, 65, 74), (90, 180, 90, 91, 300),
         (24, 48, 24, 25, 2600), (181, 360, 90, 91, 384), (240, 480, 240, 241, 160), (361, 720, 361, 361, 73)]


@pytest.mark.parametrize("nlat,nlon,lmax,mmax,rows", CASES)
@pytest.mark.parametrize("shift", [0, 1])
def test_legendre_stage(lib_built, nlat, nlon, lmax, mmax, rows, shift):
    import makani_amd as ma
    from makani_amd._lib import check, lib
    from makani_amd.sht import _stream_ptr, legendre_table, quadrature

    print(f"case Legendre stage {nlat}x{nlon} lmax={lmax} mmax={mmax} rows={rows} shift={shift}", flush=True)
    dev = torch.device("cuda", 0)
    fwd, inv = ma.RealSHT(nlat, nlon, lmax=lmax, mmax=mmax, grid="equiangular"), ma.InverseRealSHT(nlat, nlon, lmax=lmax, mmax=mmax, grid="equiangular")
    p, q = fwd.plan(dev).handle, inv.plan(dev).handle
    s = _stream_ptr(dev)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    theta, w = quadrature("equiangular", nlat)
    ld = int(lib.sfno_spectral_ld(rows))
    gen = torch.Generator().manual_seed(rows)
    magnitude = torch.exp2(torch.randint(-60, 60, (1, 1, ld), generator=gen).float())

    def buffer(n):
        """n floats that begin `shift` floats past a 16-byte boundary"""
        return torch.full((n + 4,), float("nan"), device="cuda")[shift:shift + n]

    def values(rows_of_k):
        x = torch.randn(mmax, rows_of_k, ld, generator=gen) * magnitude
        x[:, rows_of_k // 2:rows_of_k // 2 + 1] *= 2.0**12        # the bound of every column moves in the middle of its range
        x[:, -1] *= 2.0**9
        x[:, :, 1::7] = 0.0
        y = buffer(x.numel()).view(x.shape)
        y.copy_(x)
        return x, y

    def compare(got, want, size, largest, what):
        # two-part operands: 2^-21 of every product, 2^-38 of the largest ones of its row and column; fp32 sums of the products
        k = size[1]
        bound = 2.0**-20 * size[0] + 2.0**-24 * np.sqrt(k) * size[0] + k * 2.0**-37 * largest + 1e-300
        err = np.abs(got.double().cpu().numpy() - want)
        assert (err <= bound).all(), f"{what}: {np.max(err / bound):.2f} of the bound"

    x, xd = values(nlat)
    spec = buffer(mmax * lmax * ld).view(mmax, lmax, ld)
    check(lib.sfno_legendre_analysis(p, ptr(xd), ptr(spec), rows, s), "analysis")
    c, cd = values(lmax)
    out = buffer(mmax * nlat * ld).view(mmax, nlat, ld)
    check(lib.sfno_legendre_synthesis(q, ptr(cd), ptr(out), rows, s), "synthesis")
    torch.cuda.synchronize()
    step = max(1, mmax // 12)
    ta, ts = legendre_table(mmax, lmax, theta), legendre_table(mmax, lmax, theta, inverse=True)
    for m in sorted({*range(0, mmax, step), 1, mmax - 1}):
        assert torch.isnan(spec[m, :min(m, lmax)]).all(), "entries above the diagonal are not written"
        if m < lmax:
            t, v = ta[m, m:] * w, x[m].double().numpy()
            compare(spec[m, m:], t @ v, (np.abs(t) @ np.abs(v), nlat), np.abs(t).max(1)[:, None] * np.abs(v).max(0), f"analysis, order {m}")
        t, v = ts[m, m:].T, c[m, m:].double().numpy()
        if m < lmax:
            compare(out[m], t @ v, (np.abs(t) @ np.abs(v), lmax), np.abs(t).max() * np.abs(v).max(0)[None], f"synthesis, order {m}")
        else:
            assert torch.equal(out[m], torch.zeros_like(out[m]))
