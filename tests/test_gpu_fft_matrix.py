"""Longitude FFT of long bfloat16 gradient rows with few orders on the matrix units (csrc/fft_matrix.hip), through the adjoint of the
synthesis, against the vector kernels on the same values in float32: every product is exact in either, an output is an fp32 sum over
N = 1152 ... 1440 terms in levels of at most 45, 8 and 4 (the vector kernels' are 16, 10 and 9), twiddles carry one fp32 rounding: both within
3 * 2^-24 * sqrt(45) < 1.2e-6 of the exact transform, 1e-6 between them here."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

# the most orders each length has the kernel for, and one more; rows that fill a group of sixteen, half of one, one and a bit
CASES = [(6, 1440, 248, 16), (3, 1440, 249, 16), (9, 1440, 241, 8), (17, 1440, 24, 37), (2, 1440, 1, 1), (5, 1280, 221, 18), (4, 1280, 222, 2), (11, 1152, 199, 7),
         (8, 1152, 37, 33), (120, 1440, 60, 40)]


@pytest.mark.parametrize("nlat,nlon,mmax,rows", CASES)
@pytest.mark.parametrize("shift", [0, 4])
def test_adjoint_synthesis(lib_built, nlat, nlon, mmax, rows, shift):
    """shift: elements by which the tensor starts off a 16-byte boundary (those calls stay with the vector kernel)."""
    import makani_amd as ma
    from makani_amd import _lib
    from makani_amd._lib import check, lib
    from makani_amd.sht import _stream_ptr

    print(f"case matrix rfft {nlat}x{nlon} mmax={mmax} rows={rows} shift={shift}", flush=True)
    lmax = mmax + 3
    inv = ma.InverseRealSHT(nlat, nlon, lmax=lmax, mmax=mmax, grid="equiangular").cuda()
    p = inv.plan(torch.device("cuda", 0), adjoint=True).handle
    x = torch.randn(rows, nlat, nlon, generator=torch.Generator().manual_seed(3)).bfloat16()
    buf = torch.zeros(x.numel() + 8, dtype=torch.bfloat16, device="cuda")
    buf[shift:shift + x.numel()] = x.flatten().cuda()
    xf = x.float().cuda()
    nbytes = int(lib.sfno_sht_workspace_bytes(p, rows))

    def run(ptr, dtype):
        spec = torch.full((mmax, lmax, int(lib.sfno_spectral_ld(rows))), float("nan"), device="cuda")
        ws = torch.full((nbytes // 4,), float("nan"), device="cuda")
        check(lib.sfno_sht_synthesis_adjoint(p, ctypes.c_void_p(ptr), dtype, ctypes.c_void_p(spec.data_ptr()), rows, ctypes.c_void_p(ws.data_ptr()), nbytes,
                                             _stream_ptr(spec.device)), "sfno_sht_synthesis_adjoint")
        torch.cuda.synchronize()
        keep = torch.arange(mmax)[:, None] <= torch.arange(lmax)[None, :]
        return spec.cpu()[keep].double()

    got, want = run(buf.data_ptr() + 2 * shift, _lib.DTYPE_BF16), run(xf.data_ptr(), _lib.DTYPE_F32)
    assert torch.isfinite(got).all()
    # row by row (an order or a row that is wrong fails by far more)
    a, b = got[:, :2 * rows].reshape(-1, rows, 2), want[:, :2 * rows].reshape(-1, rows, 2)
    assert float((torch.linalg.norm(a - b, dim=(0, 2)) / torch.linalg.norm(b, dim=(0, 2))).max()) < 1e-6
    assert got.shape[1] == 2 * rows or float(got[:, 2 * rows:].abs().max()) == 0.0 or shift or (nlon, mmax) in ((1440, 249), (1280, 222))
