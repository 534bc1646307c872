"""The longitude transforms where the last batch of channel pairs is not full: every remainder of the batches of eight and of four pairs, odd row counts, all orders
kept and a truncated plan, the difference of two fields, against float64."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# (nlon, mmax): batches of eight pairs (96, 360), and of four that share tiles of eight (1024 and 1440; the truncated inverse takes both at once)
LENGTHS = [(96, 49), (360, 100), (1024, 513), (1440, 721), (1440, 200)]


@pytest.mark.parametrize("nlon,mmax", LENGTHS)
@pytest.mark.parametrize("rows", [1, 2, 3, 6, 7, 8, 9, 11, 14, 15, 17, 25, 32, 33])
def test_ragged_batches(lib_built, nlon, mmax, rows):
    import makani_amd as ma
    from makani_amd._lib import check, lib
    from makani_amd.sht import _stream_ptr

    print(f"case ragged FFT nlon={nlon} mmax={mmax} rows={rows}", flush=True)
    nlat, lmax = 18, 18                                  # (more latitudes than XCDs, an odd number on some)
    dev = torch.device("cuda", 0)
    fwd, inv = ma.RealSHT(nlat, nlon, lmax=lmax, mmax=mmax, grid="equiangular"), ma.InverseRealSHT(nlat, nlon, lmax=lmax, mmax=mmax, grid="equiangular")
    p, q = fwd.plan(dev).handle, inv.plan(dev).handle
    s = _stream_ptr(dev)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    ld = int(lib.sfno_spectral_ld(rows))
    gen = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, nlat, nlon, generator=gen)
    # a float32 FFT of N points: log2 N rounded stages, errors relative to the pair's norm; 4 of them cover the passes' products
    tol = 4 * torch.log2(torch.tensor(float(nlon))).item() * 2.0**-24

    xm = torch.full((mmax, nlat, ld), float("nan"), device="cuda")
    xd = x.cuda()
    check(lib.sfno_rfft(p, ptr(xd), 0, ptr(xm), rows, s), "sfno_rfft")
    torch.cuda.synchronize()
    ref = 2 * torch.pi / nlon * torch.fft.rfft(x.double())[..., :mmax]
    got = torch.view_as_complex(xm[..., :2 * rows].reshape(mmax, nlat, rows, 2).cpu().double()).permute(2, 1, 0)
    assert float((got - ref).norm() / ref.norm()) < tol
    # columns of pairs that are not there (that of a missing second row of a pair holds the first one's rounding errors)
    assert bool((xm[..., 4 * ((rows + 1) // 2):] == 0).all())

    c = torch.randn(rows, nlat, mmax, 2, generator=gen)
    xm = torch.full((mmax, nlat, ld), float("nan"), device="cuda")
    xm[..., :2 * rows] = c.permute(2, 1, 0, 3).reshape(mmax, nlat, 2 * rows).cuda()
    y = torch.full((rows, nlat, nlon), float("nan"), device="cuda")
    check(lib.sfno_irfft(q, ptr(xm), ptr(y), 0, rows, s), "sfno_irfft")
    torch.cuda.synchronize()
    z = torch.view_as_complex(c.double())
    z[..., 0].imag.zero_()
    if mmax == nlon // 2 + 1:
        z[..., -1].imag.zero_()
    ref = torch.fft.irfft(z, n=nlon, norm="forward")
    assert float((y.cpu().double() - ref).norm() / ref.norm()) < tol

    # the difference of two fields, transformed as it is formed
    x2 = torch.randn(rows, nlat, nlon, generator=gen).cuda()
    there = (torch.arange(lmax)[None, :] >= torch.arange(mmax)[:, None]).cuda()      # (the layout's other degrees are not written)
    assert torch.equal(fwd.analysis_diff(xd, x2)[there], fwd.analysis(xd - x2)[there])
