"""The relative H1 loss takes the fields prd - tar and tar through one Legendre stage: norms and gradient against the two transforms one after the other, for rows
that end inside a line, a batch of pairs and a pair, one or two batches of pairs per tile, and a target that needs its gradient."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nlat,nlon,batch,channels", [(9, 16, 1, 1), (17, 32, 2, 4), (17, 32, 3, 3), (33, 64, 1, 16), (21, 40, 1, 17), (9, 1440, 2, 4), (12, 1024, 1, 21), (60, 120, 2, 37)])
@pytest.mark.parametrize("squared", [False, True])
def test_pair_matches_separate_transforms(lib_built, nlat, nlon, batch, channels, squared):
    import makani_amd as ma
    from makani_amd import losses

    print(f"case h1 pair {nlat}x{nlon} batch={batch} channels={channels} squared={squared}", flush=True)
    gen = torch.Generator().manual_seed(nlat * nlon + channels)
    loss = ma.GeometricH1Loss((nlat, nlon), squared=squared, reduction=False).cuda()
    tar = torch.randn(batch, channels, nlat, nlon, generator=gen)
    prd = (tar + 0.3 * torch.randn(batch, channels, nlat, nlon, generator=gen)).cuda().requires_grad_()
    tar = tar.cuda()
    d, n = loss._norm_pair(prd, tar)
    assert type(d.grad_fn).__name__ == "_PairNormsFnBackward" and not n.requires_grad
    want_d, want_n = loss._norms(prd, tar), loss._norms(tar)
    # the columns of a transform do not depend on their neighbours, the powers of an example are summed in one order: the same numbers
    assert torch.equal(d, want_d) and torch.equal(n, want_n)
    g = torch.randn(batch, generator=gen).cuda()
    assert torch.equal(torch.autograd.grad((d / n * g).sum(), prd)[0], torch.autograd.grad((want_d / want_n * g).sum(), prd)[0])
    # a target that is differentiated goes through both transforms
    tar.requires_grad_()
    r = loss(prd, tar)
    assert torch.autograd.grad(r.sum(), tar)[0].abs().max() > 0
    with torch.no_grad():
        assert torch.equal(loss(prd, tar), (want_d / want_n).detach())


@pytest.mark.parametrize("nlat,nlon,batch,channels", [(60, 120, 2, 37), (90, 180, 1, 21), (90, 180, 1, 3)])
def test_memory_is_that_of_separate_transforms(lib_built, nlat, nlon, batch, channels):
    """What the forward keeps for the backward is the coefficients of prd - tar, and a step's peak is no higher than that of the transforms one after the other."""
    import makani_amd as ma

    print(f"case h1 pair memory {nlat}x{nlon} batch={batch} channels={channels}", flush=True)
    loss = ma.GeometricH1Loss((nlat, nlon), reduction=False).cuda()
    tar = torch.randn(batch, channels, nlat, nlon, device="cuda")
    prd = torch.randn_like(tar).requires_grad_()

    def memory(norms):
        torch.autograd.grad(norms()[0].sum(), prd)          # (plans and tables exist from here on)
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        out = norms()
        kept = torch.cuda.memory_allocated() - before
        torch.autograd.grad(out[0].sum(), prd)
        return kept, torch.cuda.max_memory_allocated() - before

    pair, apart = memory(lambda: loss._norm_pair(prd, tar)), memory(lambda: (loss._norms(prd, tar), loss._norms(tar)))
    # (small tensors take 512 bytes each)
    assert pair[0] <= apart[0] + 4096 and pair[1] <= apart[1] + 4096, (pair, apart)


@pytest.mark.parametrize("compute", ["fp32", "fp32_bf16x3", "fp32_mfma", "bf16"])
@pytest.mark.parametrize("nlat,nlon,batch,channels", [(17, 32, 3, 3), (21, 40, 1, 5), (33, 64, 1, 19), (60, 120, 2, 37), (121, 240, 3, 17)])
def test_pair_in_every_table_format(lib_built, compute, nlat, nlon, batch, channels):
    """Columns of one tile that belong to either field, in the kernels of every compute mode: the bits of separate transforms."""
    import makani_amd as ma

    print(f"case h1 pair {compute} {nlat}x{nlon} batch={batch} channels={channels}", flush=True)
    loss = ma.GeometricH1Loss((nlat, nlon), reduction=False).cuda()
    loss.sht = ma.RealSHT(nlat, nlon, grid="equiangular", compute=compute)
    tar = torch.randn(batch, channels, nlat, nlon, device="cuda")
    prd = torch.randn_like(tar).requires_grad_()
    d, n = loss._norm_pair(prd, tar)
    assert type(d.grad_fn).__name__ == "_PairNormsFnBackward"
    want_d, want_n = loss._norms(prd, tar), loss._norms(tar)
    assert torch.equal(d, want_d) and torch.equal(n, want_n)
    assert torch.equal(torch.autograd.grad(d.sum(), prd)[0], torch.autograd.grad(want_d.sum(), prd)[0])
