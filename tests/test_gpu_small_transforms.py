"""Small transforms exchange coefficients in the reference layout with the Legendre kernel itself; the results are those of the spectral layout and
its layout pass, bit for bit, zeros above the diagonal included."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# one column tile and several, remainders of the row blocks of 32, one degree, one order, an order past the last degree, the largest sizes
# of the direct route and sizes past it
CASES = [(32, 64, 32, 33, 8), (8, 16, 8, 9, 1), (33, 64, 33, 33, 61), (16, 32, 5, 6, 3), (40, 80, 40, 12, 37), (64, 128, 64, 64, 31), (12, 24, 7, 1, 5),
         (12, 24, 1, 2, 5), (66, 132, 65, 66, 2), (32, 64, 32, 32, 128), (32, 64, 32, 32, 129), (32, 64, 32, 32, 256), (32, 64, 32, 32, 257), (16, 32, 4, 9, 3)]


@pytest.mark.parametrize("nlat,nlon,lmax,mmax,rows", CASES)
def test_same_bits_as_the_layout_pass(lib_built, nlat, nlon, lmax, mmax, rows):
    import makani_amd as ma
    from makani_amd import _lib
    from makani_amd._lib import check, lib
    from makani_amd.sht import _stream_ptr

    print(f"case small transform {nlat}x{nlon} lmax={lmax} mmax={mmax} rows={rows}", flush=True)
    fwd = ma.RealSHT(nlat, nlon, lmax=lmax, mmax=mmax, grid="equiangular").cuda()
    inv = ma.InverseRealSHT(nlat, nlon, lmax=lmax, mmax=mmax, grid="equiangular").cuda()
    dev = torch.device("cuda", 0)
    p, q = fwd.plan(dev).handle, inv.plan(dev).handle
    s = _stream_ptr(dev)
    x = torch.randn(rows, nlat, nlon, generator=torch.Generator().manual_seed(5)).cuda()
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    nbytes = max(int(lib.sfno_sht_workspace_bytes(p, rows)), int(lib.sfno_sht_workspace_bytes(q, rows)))
    ws = torch.full((nbytes // 4 + 4,), float("nan"), device="cuda")
    spec = torch.full((mmax, lmax, int(lib.sfno_spectral_ld(rows))), float("nan"), device="cuda")
    got = torch.full((rows, lmax, mmax, 2), float("nan"), device="cuda")
    want = got.clone()
    check(lib.sfno_sht_forward(p, ptr(x), ptr(got), rows, ptr(ws), nbytes, s), "forward")
    check(lib.sfno_sht_analysis(p, ptr(x), _lib.DTYPE_F32, ptr(spec), rows, ptr(ws), nbytes, s), "analysis")
    check(lib.sfno_spectral_to_coeffs(ptr(spec), ptr(want), rows, lmax, mmax, 1, s), "layout")
    torch.cuda.synchronize()
    assert torch.isfinite(got).all() and torch.equal(got, want)
    assert float(torch.view_as_complex(got).triu(1).abs().max()) == 0.0

    # values above the diagonal are not read
    c = torch.view_as_complex(got) + torch.triu(torch.full((lmax, mmax), 7.0, device="cuda"), 1)
    c = c.contiguous()
    y, z = torch.full_like(x, float("nan")), torch.full_like(x, float("nan"))
    check(lib.sfno_sht_inverse(q, ptr(c), ptr(y), rows, ptr(ws), nbytes, s), "inverse")
    check(lib.sfno_coeffs_to_spectral(ptr(c), ptr(spec), rows, lmax, mmax, 1, s), "layout")
    check(lib.sfno_sht_synthesis(q, ptr(spec), ptr(z), _lib.DTYPE_F32, rows, ptr(ws), nbytes, s), "synthesis")
    torch.cuda.synchronize()
    assert torch.isfinite(y).all() and torch.equal(y, z)
