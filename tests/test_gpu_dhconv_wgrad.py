"""Weight gradient of dhconv (csrc/dhconv_wgrad.hip) at the sizes where its tiles and row chunks can go wrong, against
the complex128 sum on the same operands.

Bound: both operands are cut exactly into three bf16 numbers (each rounded to nearest: 2^-8, 2^-16 of the value at worst) and the
partial products left out are below 2^-23 of a product, whatever its operands' magnitudes; the sums are 12 K / 16 fp32 additions,
each off by 2^-24 at worst, on average by half of that and with either sign: 0.5 sqrt(12 K / 16) 2^-24 = 8.6e-7 in relative L2
for the K <= 1100 rows here, 1.5e-6 asserted.
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "B,I,O,L,M,triangular",
    [
        (1, 1, 1, 1, 1, True),
        (1, 32, 32, 8, 8, False),       # one tile, rows a half chunk
        (2, 33, 31, 9, 7, False),       # fewer than 8 orders: two samples per chunk
        (5, 20, 33, 12, 5, True),       # an odd number of them
        (3, 96, 64, 24, 8, False),
        (3, 31, 33, 17, 15, True),      # the second half of a chunk overlaps the first
        (1, 64, 65, 20, 16, True),      # exactly one chunk
        (2, 65, 64, 31, 17, True),      # the last chunk starts early
        (4, 40, 96, 50, 270, False),    # many chunks per sample, rectangle
        (1, 520, 519, 60, 61, True),    # 32 x 32 tiles, many of them
        (1, 648, 641, 60, 61, True),    # 64 x 64 tiles (enough of them for every CU)
    ],
)
def test_weight_grad_edges(lib_built, B, I, O, L, M, triangular):
    from makani_amd.contractions import _to_spectral, _weight_grad

    print(f"case wgrad B={B} I={I} O={O} L={L} M={M} tri={triangular}", flush=True)
    gen = torch.Generator().manual_seed(3)
    x, g = (torch.randn(B, c, L, M, dtype=torch.complex64, generator=gen) for c in (I, O))
    # magnitudes that grow or fall along the orders and jump between samples, in opposite directions for the two operands so that
    # every chunk counts in the sum
    slope, jump = min(0.5, 16 / M) * torch.arange(M), 6.0 * torch.arange(B).reshape(B, 1, 1, 1)
    x = (x * 2.0 ** (slope - jump)).cuda()
    g = (g * 2.0 ** (torch.randint(-20, 20, (1, O, 1, 1), generator=gen) - slope + jump)).cuda()
    sx, sg = _to_spectral(x, B * I, L, M, triangular), _to_spectral(g, B * O, L, M, triangular)
    keep = torch.ones(L, M, dtype=torch.bool, device="cuda")
    if triangular:
        keep = torch.arange(M, device="cuda")[None, :] <= torch.arange(L, device="cuda")[:, None]
        for s in (sx, sg):                       # orders above the degree are never read
            s[~keep.t()] = float("nan")
    got = _weight_grad(sx, sg, (I, O, L), B, M, triangular).to(torch.complex128)
    torch.cuda.synchronize()
    xl = (x.to(torch.complex128) * keep).permute(2, 1, 0, 3).reshape(L, I, B * M).contiguous()
    gl = (g.to(torch.complex128) * keep).permute(2, 0, 3, 1).reshape(L, B * M, O).contiguous()
    ref = torch.bmm(xl.conj().resolve_conj(), gl).permute(1, 2, 0)
    err = (got - ref).norm(dim=0) / ref.norm(dim=0).clamp_min(1e-300)      # per output channel and degree: each has its own scale
    assert torch.isfinite(torch.view_as_real(got)).all()
    assert float(err.max()) < 1.5e-6


@pytest.mark.parametrize("bits", [15, 22, 40])
@pytest.mark.parametrize("B,I,O,L,M,triangular", [(2, 48, 40, 24, 100, False), (1, 648, 641, 60, 61, True)])
def test_orders_of_any_magnitude_count(lib_built, B, I, O, L, M, triangular, bits):
    """x rises by 2^bits within 16 consecutive orders where g falls by as much, so that the smallest values of either count as much as the
    largest; the first 16 orders are another 2^6 off.  The bound is the one above: fp32 arithmetic does not see such a range."""
    from makani_amd.contractions import _to_spectral, _weight_grad

    print(f"case wgrad range B={B} I={I} O={O} L={L} M={M} tri={triangular} bits={bits}", flush=True)
    gen = torch.Generator().manual_seed(5)
    x, g = (torch.randn(B, c, L, M, dtype=torch.complex64, generator=gen) for c in (I, O))
    m = torch.arange(M)
    ramp = 2.0 ** (bits * (m % 16) / 15.0 + 6.0 * (m < 16))
    x, g = (x * ramp).cuda(), (g / ramp).cuda()
    got = _weight_grad(_to_spectral(x, B * I, L, M, triangular), _to_spectral(g, B * O, L, M, triangular), (I, O, L), B, M, triangular).to(torch.complex128)
    keep = torch.ones(L, M, dtype=torch.bool, device="cuda")
    if triangular:
        keep = torch.arange(M, device="cuda")[None, :] <= torch.arange(L, device="cuda")[:, None]
    xl = (x.to(torch.complex128) * keep).permute(2, 1, 0, 3).reshape(L, I, B * M).contiguous()
    gl = (g.to(torch.complex128) * keep).permute(2, 0, 3, 1).reshape(L, B * M, O).contiguous()
    ref = torch.bmm(xl.conj().resolve_conj(), gl).permute(1, 2, 0)
    err = (got - ref).norm(dim=0) / ref.norm(dim=0).clamp_min(1e-300)
    assert float(err.max()) < 1.5e-6


def test_row_strides_beyond_32_bits(lib_built):
    """16 row strides of more than 4 GiB (one order, 66048 rows of 512 degrees): 64-bit offsets.  516 chunks of two samples make 12 * 516
    additions: 0.5 sqrt(6192) 2^-24 = 2.4e-6 by the reckoning above, asserted."""
    from makani_amd.contractions import _to_spectral, _weight_grad

    B, I, O, L, M = 1032, 64, 33, 512, 1
    print("case wgrad 64-bit offsets", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(6)
    x, g = (torch.view_as_complex(torch.randn(B, c, L, M, 2, device="cuda", generator=gen)) for c in (I, O))
    sx, sg = _to_spectral(x, B * I, L, M, True), _to_spectral(g, B * O, L, M, True)
    assert 64 * L * max(sx.shape[-1], sg.shape[-1]) > 2 ** 32
    got = _weight_grad(sx, sg, (I, O, L), B, M, True)
    torch.cuda.synchronize()
    for l in (0, 1, 7, 8, 255, 511):
        ref = torch.matmul(x[:, :, l, 0].to(torch.complex128).t().conj().resolve_conj().contiguous(), g[:, :, l, 0].to(torch.complex128).contiguous())
        err = (got[:, :, l].to(torch.complex128) - ref).norm(dim=0) / ref.norm(dim=0)
        assert float(err.max()) < 2.4e-6, l


@pytest.mark.parametrize("I,O,L", [(256, 200, 333), (600, 610, 49)])
def test_weights_packed_in_slabs_of_degrees(lib_built, I, O, L):
    """Weights above 96 MB are packed a slab of degrees at a time (here two slabs, the last one shorter and no multiple of 16): output and
    input gradient of two rows per degree against complex128, with the bound above (K <= 610)."""
    from makani_amd.contractions import _contract_dhconv

    print(f"case slabs {I} {O} {L}", flush=True)
    gen = torch.Generator().manual_seed(3)
    w = torch.randn(I, O, L, dtype=torch.complex64, generator=gen) * torch.logspace(-3, 3, L)
    x = torch.randn(1, I, L, 2, dtype=torch.complex64, generator=gen)
    g = torch.randn(1, O, L, 2, dtype=torch.complex64, generator=gen)
    xd = x.cuda().requires_grad_()
    y = _contract_dhconv(xd, w.cuda())
    y.backward(g.cuda())
    # per degree, so that every slab counts alike
    wl, xl, gl = (t.to(torch.complex128) for t in (w.permute(2, 0, 1), x[0].permute(1, 2, 0), g[0].permute(1, 2, 0)))
    for got, ref in ((y.detach(), torch.matmul(xl, wl)), (xd.grad, torch.matmul(gl, wl.conj().transpose(1, 2)))):
        d = got[0].cpu().permute(1, 2, 0).to(torch.complex128) - ref
        assert float((d.abs().square().sum((1, 2)) / ref.abs().square().sum((1, 2))).max()) ** 0.5 < 1.5e-6


@pytest.mark.parametrize("L", [5, 16, 50, 72])
@pytest.mark.parametrize("I,O", [(64, 20), (70, 40), (130, 33)])
def test_units_of_half_a_group(lib_built, L, I, O):
    """One to nine groups of degrees whose tiles (an even and odd number of input blocks) are dealt to the XCDs whole or in halves."""
    from makani_amd.contractions import _to_spectral, _weight_grad

    print(f"case wgrad units L={L} I={I} O={O}", flush=True)
    gen = torch.Generator().manual_seed(L)
    x, g = (torch.randn(2, c, L, L, dtype=torch.complex64, generator=gen).tril().cuda() for c in (I, O))
    got = _weight_grad(_to_spectral(x, 2 * I, L, L, True), _to_spectral(g, 2 * O, L, L, True), (I, O, L), 2, L, True).to(torch.complex128)
    torch.cuda.synchronize()
    xl, gl = (t.to(torch.complex128).permute(2, 0, 3, 1).reshape(L, 2 * L, -1).contiguous() for t in (x, g))
    ref = torch.bmm(xl.transpose(1, 2).conj().resolve_conj().contiguous(), gl).permute(1, 2, 0)
    assert float((got - ref).norm() / ref.norm()) < 1.5e-6
