"""norm -> GELU -> 1x1 convolution -> GELU -> 1x1 convolution in one kernel (csrc/pointwise_mlp.h) against float64 on the same bf16 operands.

Bound: the two intermediate fields are rounded to bf16 in the oracle as in the kernel, so what differs is fp32 sums of at most 768 bf16
products (1e-6 relative), the GELU's fit (7e-5 of its tail) and values that round the other way for it (one in a hundred, by one bf16 step:
2^-8 * sqrt(0.01) = 4e-4 of the field), and the rounding of the result (1.7e-3 on average): 2^-8 in relative L2; element-wise 2^-7 of
the value plus 2^-7 of the field's scale.  Against the three kernels it replaces: the same bits."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def operands(B, E, hidden, H, W, bias):
    gen = torch.Generator().manual_seed(17)
    x = (2.0 * torch.randn(B, E, H, W, generator=gen) + 1.0).bfloat16()
    sc, sh = 0.5 + torch.rand(B, E, generator=gen), torch.randn(B, E, generator=gen)
    w1, w2 = torch.randn(hidden, E, 1, 1, generator=gen) / E ** 0.5, torch.randn(E, hidden, 1, 1, generator=gen) / hidden ** 0.5
    b1, b2 = (torch.randn(hidden, generator=gen), torch.randn(E, generator=gen)) if bias else (None, None)
    return [t.cuda() if t is not None else None for t in (x, sc, sh, w1, b1, w2, b2)]


def oracle(x, sc, sh, w1, b1, w2, b2):
    def conv(w, v, b):
        y = torch.matmul(w.bfloat16().double().flatten(1), v.bfloat16().double().flatten(2))
        return (y if b is None else y + b.double()[:, None]).reshape(v.shape[0], w.shape[0], *v.shape[2:])

    h = F.gelu(x.double() * sc.double()[..., None, None] + sh.double()[..., None, None])
    return conv(w2, F.gelu(conv(w1, h, b1)), b2)


@pytest.mark.parametrize(
    "B,E,hidden,H,W,bias",
    [
        (1, 8, 16, 1, 8, True), (2, 32, 64, 4, 8, True), (1, 64, 128, 9, 16, False),           # one chunk of hidden channels, part of a tile
        (2, 104, 208, 16, 24, True), (1, 128, 256, 32, 64, True), (3, 136, 272, 11, 24, True),  # ragged steps, 128 and 256 rows
        (1, 256, 512, 30, 60, False), (1, 264, 400, 23, 40, True), (2, 384, 768, 33, 64, True),
        (1, 384, 576, 200, 360, True), (1, 72, 80, 181, 360, True),                            # several tiles per workgroup, the last one ragged
    ],
)
def test_norm_mlp(lib_built, B, E, hidden, H, W, bias):
    from makani_amd import pointwise as pw

    print(f"case norm_mlp B={B} {E}->{hidden}->{E} {H}x{W}", flush=True)
    ops = operands(B, E, hidden, H, W, bias)
    got, want = pw.norm_mlp(*ops).double(), oracle(*ops)
    assert float((got - want).norm() / want.norm()) < 2 ** -8
    assert float(((got - want).abs() / (want.abs() + want.std())).max()) < 2 ** -7
    # the three kernels form the same sums in the same order
    x, sc, sh, w1, b1, w2, b2 = ops
    three = pw.conv1x1(pw.conv1x1(pw.scale_shift_act(x, sc, sh, "gelu"), w1, b1, "gelu"), w2, b2)
    assert torch.equal(got, three.double())


def test_in_place_and_nan(lib_built):
    """The result may overwrite the input (every tile is read before it is written), and a NaN or an infinity stays within its pixel."""
    import ctypes

    from makani_amd import pointwise as pw
    from makani_amd._lib import check, lib

    B, E, hidden, H, W = 2, 136, 272, 90, 184          # two tiles for some workgroups, rows and steps past the matrices
    x, sc, sh, w1, b1, w2, b2 = operands(B, E, hidden, H, W, True)
    want = pw.norm_mlp(x, sc, sh, w1, b1, w2, b2)
    p = [ctypes.c_void_p(t.data_ptr()) for t in (sc, sh, pw.packed_weight(w1), b1, pw.packed_weight(w2), b2)]
    y = x.clone()
    check(lib.sfno_pointwise_mlp(ctypes.c_void_p(y.data_ptr()), *p, ctypes.c_void_p(y.data_ptr()), B, E, hidden, H * W, pw._stream(x.device)), "sfno_pointwise_mlp")
    assert torch.equal(y, want)
    x[0, 5, 3, 7], x[1, E - 1, 80, 100] = float("nan"), float("inf")
    got = pw.norm_mlp(x, sc, sh, w1, b1, w2, b2)
    bad = torch.zeros_like(got, dtype=torch.bool)
    bad[0, :, 3, 7] = bad[1, :, 80, 100] = True
    assert torch.equal(got[~bad], want[~bad]) and bool(got[0, :, 3, 7].isnan().all()) and not bool(got[1, :, 80, 100].isfinite().any())


def test_refusals(lib_built):
    """Outside its range the call is refused, not run: sizes it has no tiles for, null pointers, tensors off 16-byte boundaries."""
    from makani_amd._lib import lib

    def call(E, hidden, P, x=16, y=16, w=16):
        return lib.sfno_pointwise_mlp(x, 16, 16, w, None, w, None, y, 1, E, hidden, P, None)

    for E, hidden, P in ((392, 768, 64), (12, 32, 64), (32, 40, 64), (32, 64, 60)):
        assert call(E, hidden, P) == -5
    assert call(32, 64, 64, x=None) == call(32, 64, 64, y=18) == call(32, 64, 64, w=24) == call(0, 64, 64) == -1
