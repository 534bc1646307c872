"""Every length with specialised FFT kernels (csrc/fft_lengths.h), along longitude and along latitude, through the planar pair
against numpy's float64 transforms.

Bound: an fp32 FFT of n points rounds each value once per base-radix stage, relative L2 error about 2^-24 sqrt(c log2 n) with c below 4
for the radices used: 4e-7 at 1536 points, two of them (longitude, latitude) below 8e-7; 1.5e-6 asserted."""
import os
import re

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu
TOL = 1.5e-6
HERE = os.path.dirname(os.path.abspath(__file__))
with open(os.path.join(HERE, "..", "modulus-makani_amd", "csrc", "fft_lengths.h")) as f:
    LENGTHS = sorted(int(n) for n in re.findall(r"X\((\d+),", f.read()))


def rel(a, b):
    return float(np.linalg.norm(np.asarray(a) - b) / np.linalg.norm(b))


def kept(nlat, lmax):
    return np.r_[0:(lmax + 1) // 2, nlat - lmax // 2:nlat]


@pytest.mark.parametrize("n", LENGTHS)
def test_longitude(lib_built, n):
    """Order-major kernels (nine latitudes have no column kernel; test_row_ordered_pair has the others)."""
    import makani_amd as ma

    print(f"case lon {n}", flush=True)
    rng = np.random.default_rng(n)
    nlat = 9
    for rows, mmax in ((5, n // 2 + 1), (18, n // 6 + 1)):       # all orders, and few of them (another kernel of the inverse)
        x = rng.standard_normal((rows, nlat, n)).astype(np.float32)
        fwd, inv = ma.RealFFT2(nlat, n, mmax=mmax), ma.InverseRealFFT2(nlat, n, mmax=mmax)
        want = np.fft.rfft2(x.astype(np.float64), norm="ortho")[..., :mmax]
        assert rel(fwd(torch.from_numpy(x).cuda()).cpu().numpy(), want) < TOL
        back = np.fft.irfft2(want, s=(nlat, n), norm="ortho")
        c = torch.from_numpy(want.astype(np.complex64)).cuda()
        assert rel(inv(c).cpu().numpy(), back) < TOL
        # bf16 fields in and out of the spectral layout, and the moments of the rows over longitude
        xb = torch.from_numpy(x).cuda().to(torch.bfloat16)
        assert torch.equal(fwd.analysis(xb), fwd.analysis(xb.float()))
        spec = fwd.analysis(torch.from_numpy(x).cuda())
        y = inv.synthesis(spec, (rows,))
        assert torch.equal(inv.synthesis(spec, (rows,), dtype=torch.bfloat16), y.to(torch.bfloat16))
        ys, stats = inv.synthesis_with_lat_stats(spec, (rows,))
        assert torch.equal(ys, y)
        yd = y.double()
        assert torch.allclose(stats[..., 0].double(), yd.mean(-1), atol=2e-6)
        assert torch.allclose(stats[..., 1].double(), yd.var(-1, unbiased=False), rtol=1e-5)


@pytest.mark.parametrize("n", [n for n in LENGTHS if n <= 1024])
def test_latitude(lib_built, n):
    import makani_amd as ma

    print(f"case lat {n}", flush=True)
    rng = np.random.default_rng(n)
    nlon, rows = 32, 3
    for lmax, mmax in ((n, 17), (n // 2 + 1, 11)):
        x = rng.standard_normal((rows, n, nlon)).astype(np.float32)
        fwd, inv = ma.RealFFT2(n, nlon, lmax=lmax, mmax=mmax), ma.InverseRealFFT2(n, nlon, lmax=lmax, mmax=mmax)
        want = np.fft.rfft2(x.astype(np.float64), norm="ortho")[:, kept(n, lmax), :mmax]
        assert rel(fwd(torch.from_numpy(x).cuda()).cpu().numpy(), want) < TOL
        full = np.zeros((rows, n, nlon // 2 + 1), dtype=complex)
        full[:, kept(n, lmax), :mmax] = want
        back = np.fft.irfft2(full, s=(n, nlon), norm="ortho")
        assert rel(inv(torch.from_numpy(want.astype(np.complex64)).cuda()).cpu().numpy(), back) < TOL


def planar_reference(x, lmax, mmax):
    """float64 coefficients of x and the field they give back"""
    nlat, n = x.shape[-2:]
    c = np.fft.rfft2(x.astype(np.float64), norm="ortho")[..., kept(nlat, lmax), :mmax]
    full = np.zeros((*x.shape[:-2], nlat, n // 2 + 1), dtype=complex)
    full[..., kept(nlat, lmax), :mmax] = c
    return c, np.fft.irfft2(full, s=(nlat, n), norm="ortho")


@pytest.mark.parametrize("n", LENGTHS)
def test_row_ordered_pair(lib_built, n):
    """Row kernels of every length, which take latitude counts with column kernels only (test_longitude has none): all orders and few of
    them, groups of 16 orders that are not full; the last tile of row pairs is not either.  Adjoints by <A x, c> = <x, A^T c>."""
    import makani_amd as ma

    print(f"case rows {n}", flush=True)
    rng = np.random.default_rng(n)
    for rows, nlat, lmax, mmax in ((5, 12, 12, n // 2 + 1), (7, 8, 5, max(2, n // 6 + 1))):
        x = rng.standard_normal((rows, nlat, n)).astype(np.float32)
        fwd, inv = ma.RealFFT2(nlat, n, lmax=lmax, mmax=mmax), ma.InverseRealFFT2(nlat, n, lmax=lmax, mmax=mmax)
        want, back = planar_reference(x, lmax, mmax)
        xd = torch.from_numpy(x).cuda().requires_grad_()
        got = fwd(xd)
        assert rel(got.detach().cpu().numpy(), want) < TOL
        cd = torch.from_numpy(want.astype(np.complex64)).cuda().requires_grad_()
        y = inv(cd)
        assert rel(y.detach().cpu().numpy(), back) < TOL
        u = (rng.standard_normal(want.shape) + 1j * rng.standard_normal(want.shape)).astype(np.complex64)
        v = rng.standard_normal(x.shape).astype(np.float32)
        got.backward(torch.from_numpy(u).cuda())
        y.backward(torch.from_numpy(v).cuda())
        # real inner products; both sides are sums of products of normal numbers: the error is TOL of the vectors' norms
        for lhs, rhs, norms in (
            (np.sum(want.real * u.real + want.imag * u.imag), np.sum(x.astype(np.float64) * xd.grad.cpu().numpy()), np.linalg.norm(want) * np.linalg.norm(u)),
            (np.sum(back * v), np.sum((want.conj() * cd.grad.cpu().numpy()).real), np.linalg.norm(back) * np.linalg.norm(v)),
        ):
            assert abs(lhs - rhs) < TOL * norms


@pytest.mark.parametrize("rows,nlat,n", [(400, 64, 96), (140, 64, 1024)])
def test_row_kernels_walk_many_tiles(lib_built, rows, nlat, n):
    """More tiles of row pairs than resident workgroups (1024 of 8 pairs, 512 of 4): the second round of the persistent loops, element by
    element.  fp32 transform pairs of normal numbers: TOL of their standard deviation, six times that at most over all elements."""
    import makani_amd as ma

    print(f"case row tiles {rows} {nlat} {n}", flush=True)
    x = np.random.default_rng(1).standard_normal((rows, nlat, n)).astype(np.float32)
    fwd, inv = ma.RealFFT2(nlat, n), ma.InverseRealFFT2(nlat, n)
    want, back = planar_reference(x, nlat, n // 2 + 1)
    assert np.abs(fwd(torch.from_numpy(x).cuda()).cpu().numpy() - want).max() < 6 * TOL
    assert np.abs(inv(torch.from_numpy(want.astype(np.complex64)).cuda()).cpu().numpy() - back).max() < 6 * TOL
