"""Transforms leave the high orders near the poles out of the Fourier buffer: the Legendre analysis does not read them, the synthesis does not write them, the
longitude kernels skip them.  Their results are those of the separate stages, which exchange the whole buffer, bit for bit, whatever the buffer held before."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# grids whose polar rows drop orders and one that drops none, truncated degrees, orders past the last degree, more orders than the longitudes resolve
# (inverse only), an even and an odd number of latitudes, lengths with one and with two batches per tile
CASES = [(32, 64, 32, 33), (181, 360, 181, 181), (180, 360, 60, 61), (240, 480, 200, 241), (361, 720, 120, 121), (480, 960, 180, 181), (721, 1440, 240, 241),
         (600, 1200, 600, 601)]


@pytest.mark.parametrize("nlat,nlon,lmax,mmax", CASES)
@pytest.mark.parametrize("rows,dtype,compute", [(5, "float32", "fp32"), (18, "bfloat16", "fp32"), (3, "float32", "fp32_bf16x3"), (4, "float32", "bf16")])
def test_same_bits_as_the_stages(lib_built, nlat, nlon, lmax, mmax, rows, dtype, compute):
    import makani_amd as ma
    from makani_amd import _lib
    from makani_amd._lib import check, lib
    from makani_amd.sht import _stream_ptr

    print(f"case polar orders {nlat}x{nlon} lmax={lmax} mmax={mmax} rows={rows} {dtype} {compute}", flush=True)
    dev = torch.device("cuda", 0)
    fwd = ma.RealSHT(nlat, nlon, lmax=lmax, mmax=mmax, grid="equiangular", compute=compute)
    inv = ma.InverseRealSHT(nlat, nlon, lmax=lmax, mmax=mmax, grid="equiangular", compute=compute)
    p, q = fwd.plan(dev).handle, inv.plan(dev).handle
    s = _stream_ptr(dev)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    dt, dcode = getattr(torch, dtype), _lib.DTYPE_BF16 if dtype == "bfloat16" else _lib.DTYPE_F32
    gen = torch.Generator().manual_seed(rows)
    x = torch.randn(rows, nlat, nlon, generator=gen).to(dt).cuda()
    ld = int(lib.sfno_spectral_ld(rows))
    nbytes = max(int(lib.sfno_sht_workspace_bytes(p, rows)), int(lib.sfno_sht_workspace_bytes(q, rows)))
    ws = torch.full((nbytes // 4 + 4,), float("nan"), device="cuda")
    xm = torch.full((mmax, nlat, ld), float("nan"), device="cuda")
    spec = torch.zeros(mmax, lmax, ld, device="cuda")
    got, want = spec.clone(), spec.clone()

    check(lib.sfno_sht_analysis(p, ptr(x), dcode, ptr(got), rows, ptr(ws), nbytes, s), "analysis")
    check(lib.sfno_rfft(p, ptr(x), dcode, ptr(xm), rows, s), "longitude")
    check(lib.sfno_legendre_analysis(p, ptr(xm), ptr(want), rows, s), "Legendre")
    torch.cuda.synchronize()
    assert torch.isfinite(xm[:, :, :2 * rows]).all(), "the longitude stage by itself writes every order"
    assert torch.isfinite(got[:, :, :2 * rows]).all() and torch.equal(got[:, :, :2 * rows], want[:, :, :2 * rows])

    ws.fill_(float("nan"))
    xm.fill_(float("nan"))
    y, z = torch.full_like(x, float("nan")), torch.full_like(x, float("nan"))
    moments = torch.full((rows, nlat, 2), float("nan"), device="cuda")
    check(lib.sfno_sht_synthesis(q, ptr(want), ptr(y), dcode, rows, ptr(ws), nbytes, s), "synthesis")
    check(lib.sfno_legendre_synthesis(q, ptr(want), ptr(xm), rows, s), "Legendre")
    check(lib.sfno_irfft(q, ptr(xm), ptr(z), dcode, rows, s), "longitude")
    torch.cuda.synchronize()
    assert torch.isfinite(xm[:, :, :2 * rows]).all(), "the Legendre stage by itself writes every row"
    assert torch.isfinite(y.float()).all() and torch.equal(y, z)
    ws.fill_(float("nan"))
    check(lib.sfno_sht_synthesis_lat_stats(q, ptr(want), ptr(y), dcode, rows, ptr(ws), nbytes, ptr(moments), s), "synthesis with moments")
    torch.cuda.synchronize()
    assert torch.equal(y, z) and torch.isfinite(moments).all()

    # adjoints: on memory full of NaN and on memory of zeros
    a, b = fwd.plan(dev, adjoint=True).handle, inv.plan(dev, adjoint=True).handle
    outs = []
    for fill in (float("nan"), 0.0):
        ws.fill_(fill)
        gx, gc = torch.full_like(x, float("nan")), torch.zeros_like(spec)
        check(lib.sfno_sht_analysis_adjoint(a, ptr(want), ptr(gx), dcode, rows, ptr(ws), nbytes, s), "adjoint of the analysis")
        ws.fill_(fill)
        check(lib.sfno_sht_synthesis_adjoint(b, ptr(x), dcode, ptr(gc), rows, ptr(ws), nbytes, s), "adjoint of the synthesis")
        torch.cuda.synchronize()
        outs.append((gx, gc[:, :, :2 * rows].contiguous()))
    assert all(torch.isfinite(t.float()).all() for t in outs[0]) and all(torch.equal(t, u) for t, u in zip(*outs))
