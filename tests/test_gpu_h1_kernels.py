"""Kernels of GeometricH1Loss that pass over no field of their own: the transform of a difference (csrc/fft_kernels.h) and the norms from
the per-degree power (csrc/degree_power.hip)."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlat,nlon,lead", [(32, 64, (2, 4)), (5, 8, (3,)), (91, 180, (2, 5)), (33, 480, (1, 9)), (9, 1440, (2, 9)), (7, 1440, (1, 16)), (8, 1024, (17,)),
                                            (9, 58, (3,))])
def test_analysis_of_a_difference(lib_built, nlat, nlon, lead):
    """The same bits as the transform of the stored difference, both gradients too (one and two batches of channel pairs per tile, odd row
    counts, tiles past the last pair; 58 points have no specialised kernel)."""
    import makani_amd as ma

    print(f"case difference {nlat}x{nlon} lead={lead}", flush=True)
    gen = torch.Generator().manual_seed(5)
    x, y = (torch.randn(*lead, nlat, nlon, generator=gen).cuda().requires_grad_() for _ in range(2))
    sht = ma.RealSHT(nlat, nlon, grid="equiangular")
    keep = torch.arange(sht.mmax).cuda()[:, None] <= torch.arange(sht.lmax).cuda()[None, :]
    got, want = sht.analysis_diff(x, y), sht.analysis(x - y)
    rows = x.numel() // (nlat * nlon)
    assert torch.equal(got[keep][:, :2 * rows], want[keep][:, :2 * rows])
    g = torch.where(keep[..., None], torch.randn(want.shape, generator=gen).cuda(), 0.0)
    a, b = torch.autograd.grad(got, (x, y), g), torch.autograd.grad(want, (x, y), g)
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])


def test_difference_of_other_tensors(lib_built):
    """What the kernel does not take goes through the stored difference: broadcast and strided tensors, bfloat16, views off 16 bytes."""
    import makani_amd as ma

    gen = torch.Generator().manual_seed(6)
    sht = ma.RealSHT(16, 32, grid="equiangular")
    x, y = (torch.randn(2, 3, 16, 32, generator=gen).cuda() for _ in range(2))
    shifted = torch.randn(2 * 3 * 16 * 32 + 1, generator=gen).cuda()[1:].view(2, 3, 16, 32)
    for p, q in ((x, y[:, :1]), (x, y.transpose(0, 1).contiguous().transpose(0, 1)), (x.bfloat16(), y.bfloat16()), (x, y.bfloat16()), (shifted, y)):
        assert torch.equal(torch.nan_to_num(sht.analysis_diff(p, q)[0]), torch.nan_to_num(sht.analysis(p - q)[0]))
    with pytest.raises(TypeError):
        sht.analysis_diff(x.double(), y.double())


@pytest.mark.parametrize("batch,channels,lmax,mmax", [(1, 1, 1, 1), (2, 3, 7, 5), (3, 1, 700, 3), (2, 37, 530, 9), (1, 73, 721, 4), (5, 129, 12, 12)])
@pytest.mark.parametrize("squared", [False, True])
def test_degree_norms(lib_built, batch, channels, lmax, mmax, squared):
    """Value and gradient against float64 (fp32 powers, sums in double: 1e-6), one and several workgroups per example, more and fewer degrees
    than threads; what stands in the padding columns and above the diagonal is never used."""
    from makani_amd._lib import lib
    from makani_amd.losses import _DegreeNormFn

    print(f"case norms {batch}x{channels} l={lmax} m={mmax}", flush=True)
    rows, alpha = batch * channels, 0.3
    gen = torch.Generator().manual_seed(rows)
    keep = torch.arange(mmax)[:, None] <= torch.arange(lmax)[None, :]
    spec = torch.full((mmax, lmax, int(lib.sfno_spectral_ld(rows))), float("nan"))
    spec[..., :2 * rows] = torch.where(keep[..., None], torch.randn(mmax, lmax, 2 * rows, generator=gen), torch.nan)
    w = torch.arange(lmax).float() * (torch.arange(lmax) + 1) + 0.5
    x = spec.cuda().requires_grad_()
    got = _DegreeNormFn.apply(x, w.cuda(), batch, channels, alpha, squared)
    g = torch.randn(batch, generator=gen)
    grad = torch.autograd.grad(got, x, g.cuda())[0].cpu()

    c = torch.where(keep[..., None], spec[..., :2 * rows], 0.0).double().requires_grad_()
    wm = torch.where(torch.arange(mmax) == 0, 1.0, 2.0).double()
    p = torch.einsum("m,mlrc->rl", wm, c.reshape(mmax, lmax, rows, 2) ** 2).reshape(batch, -1, lmax)
    a, h = p.sum((1, 2)), (p * w.double()).sum((1, 2))
    want = alpha * a + (1 - alpha) * h if squared else alpha * a.sqrt() + (1 - alpha) * h.sqrt()
    (gc,) = torch.autograd.grad(want, c, g.double())
    want = want.detach()
    assert float((got.detach().cpu().double() - want).norm() / want.norm()) < 1e-6
    inside = grad[keep]
    assert (inside[:, 2 * rows:] == 0).all()
    assert float((inside[:, :2 * rows].double() - gc[keep]).norm() / gc.norm()) < 1e-6
