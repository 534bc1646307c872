"""1x1 convolution at the edges of its tile choices (csrc/pointwise.hip: 128, 256 or 384 output channels per workgroup, small
tiles where the large ones would leave CUs idle), against float64 on the same bf16 operands.

Bound: fp32 sums of at most 130 bf16 products (1e-6) and one rounding to bf16, half a unit of 8 significant bits: 2^-8 of a value
at worst, so 2^-8 in relative L2 for any number of values (1.7e-3 on average); element-wise 2^-7 asserted, for the small values of a
GELU or a sum with 0.05 beside the value (their absolute error is that of the terms).
"""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "B,K,O,H,W",
    [
        (1, 5, 97, 2, 4), (1, 64, 128, 16, 16), (2, 65, 129, 8, 33),      # few pixels: one block of 128
        (1, 33, 256, 184, 240), (1, 96, 257, 176, 256),                     # 172 tiles of 256: two row tiles per wavefront; 257: 384
        (1, 31, 384, 96, 264), (1, 32, 384, 344, 128), (1, 40, 512, 176, 128), (2, 24, 640, 120, 120),
        (1, 3, 1, 1, 8), (1, 130, 96, 33, 64), (3, 64, 33, 16, 24), (2, 70, 96, 257, 512),      # at most 96: two and eight wavefronts
    ],
)
def test_tiles(lib_built, B, K, O, H, W):
    from makani_amd import pointwise as pw

    print(f"case conv {B} {K}->{O} {H}x{W}", flush=True)
    gen = torch.Generator().manual_seed(5)
    x = torch.randn(B, K, H, W, generator=gen).cuda().to(torch.bfloat16)
    w = (torch.randn(O, K, generator=gen) / K ** 0.5).cuda()
    bias = torch.randn(O, generator=gen).cuda()
    add = torch.randn(B, O, H, W, generator=gen).cuda().to(torch.bfloat16)
    sc, sh = torch.randn(B, O, generator=gen).cuda(), torch.randn(B, O, generator=gen).cuda()
    lin = torch.matmul(w.to(torch.bfloat16).double(), x.double().reshape(B, K, H * W)).reshape(B, O, H, W) + bias.double()[None, :, None, None]
    aff = sc.double()[..., None, None] * add.double() + sh.double()[..., None, None]
    for act, addend, want in ((None, None, lin), ("gelu", None, torch.nn.functional.gelu(lin)), (None, add, lin + aff)):
        got = pw.conv1x1(x, w, bias, act, addend, sc if addend is not None else None, sh if addend is not None else None).double()
        assert float((got - want).norm() / want.norm()) < 2 ** -8
        assert float(((got - want).abs() / (want.abs() + 0.05)).max()) < 2 ** -7


@pytest.mark.parametrize("K,O,H,W", [(24, 40, 16, 24), (40, 150, 24, 40), (33, 384, 40, 64)])
def test_sums_in_place(lib_built, K, O, H, W):
    """The addend may be the output, and scale_shift_act may write where it reads: bit for bit the results of separate tensors."""
    import ctypes

    from makani_amd import pointwise as pw
    from makani_amd._lib import check, lib

    print(f"case in place {K}->{O}", flush=True)
    gen = torch.Generator().manual_seed(6)
    x, add = torch.randn(2, K, H, W, generator=gen).cuda().to(torch.bfloat16), torch.randn(2, O, H, W, generator=gen).cuda().to(torch.bfloat16)
    w, sc, sh = torch.randn(O, K, generator=gen).cuda(), torch.randn(2, O, generator=gen).cuda(), torch.randn(2, O, generator=gen).cuda()
    want, act = pw.conv1x1(x, w, None, None, add, sc, sh), pw.scale_shift_act(add, sc, sh, "gelu")

    def p(t):
        return ctypes.c_void_p(t.data_ptr())

    packed, y, z = pw.packed_weight(w), add.clone(), add.clone()
    check(lib.sfno_pointwise_conv(p(x), p(packed), None, p(y), 2, K, O, H * W, 0, p(y), p(sc), p(sh), pw._stream(x.device)), "sfno_pointwise_conv")
    check(lib.sfno_scale_shift_act(p(z), p(sc), p(sh), p(z), 2 * O, H * W, 1, pw._stream(x.device)), "sfno_scale_shift_act")
    assert torch.equal(y, want) and torch.equal(z, act)
