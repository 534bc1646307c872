"""The training GELU and its derivative by table (convolutions of more than 96 output channels, one to three row tiles per wavefront) against the formulas that narrower
convolutions evaluate: the derivative at every bf16 value, the activation at every finite one through the product and at infinities, NaN and every exponent through the bias, the same bits and
NaN at the same places; and the layers that take the formula all the same."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


def _both(channels, z):
    from makani_amd import pointwise as pw
    from makani_amd._lib import check, lib

    n = z.numel()
    P = (-(-n // channels) + 7) // 8 * 8
    x = torch.zeros(channels * P, dtype=torch.bfloat16)
    x[:n] = z
    x = x.reshape(1, channels, 1, P).cuda()
    finite = torch.where(torch.isfinite(x), x, torch.zeros_like(x))          # (an infinity would meet the zeros of the identity)
    eye, ones = torch.eye(channels, device="cuda"), torch.ones_like(x)
    y, pre, gx = (torch.empty_like(x) for _ in range(3))
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    check(lib.sfno_pointwise_conv_gelu(ptr(finite), ptr(pw.packed_weight(eye)), None, ptr(y), ptr(pre), 1, channels, channels, P, pw._stream(x.device)), "forward")
    check(lib.sfno_pointwise_conv_gelu_grad(ptr(ones), ptr(pw.packed_weight(eye, transposed=True)), ptr(x), ptr(gx), 1, channels, channels, P,
                                            pw._stream(x.device)), "backward")
    torch.cuda.synchronize()
    return y.reshape(-1)[:n].cpu(), gx.reshape(-1)[:n].cpu()


@pytest.mark.parametrize("channels", [97, 128, 200, 300, 384])
def test_table_is_the_formula(lib_built, channels):
    print(f"case gelu table {channels}", flush=True)
    z = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    (y0, g0), (y1, g1) = _both(64, z), _both(channels, z)
    # (half of a subnormal number is a rounding boundary: the formula's 0.5 is off by 4e-10, the table's straight line is not)
    big = ~(z.abs() < 2.0**-120)
    assert torch.equal(y0[big].view(torch.int16), y1[big].view(torch.int16))
    assert torch.equal(torch.isnan(g0), torch.isnan(g1))
    ok = ~torch.isnan(g0)
    assert torch.equal(g0[ok].view(torch.int16), g1[ok].view(torch.int16))


@pytest.mark.parametrize("channels", [97, 128, 200, 300, 384])
def test_every_value_through_the_bias(lib_built, channels):
    """Infinities and NaN reach the activation by the bias (in the product they would meet the other weights' zeros)."""
    from makani_amd import pointwise as pw
    from makani_amd._lib import check, lib

    print(f"case gelu table, bias {channels}", flush=True)
    x = torch.zeros(1, 8, 8, dtype=torch.bfloat16, device="cuda")
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())

    def activations(O, values):
        """of `values` [n], n a multiple of O: pixel 0 of O channels with these biases, call by call"""
        w = pw.packed_weight(torch.zeros(O, 8, device="cuda"))
        ys, zs = [], []
        for b in values.split(O):
            y, z = (torch.empty(O, 8, dtype=torch.bfloat16, device="cuda") for _ in range(2))
            check(lib.sfno_pointwise_conv_gelu(ptr(x), ptr(w), ptr(b), ptr(y), ptr(z), 1, 8, O, 8, pw._stream(x.device)), "forward")
            ys.append(y[:, 0])
            zs.append(z[:, 0])
        return torch.cat(ys).cpu(), torch.cat(zs).cpu()

    # every exponent of either sign with a few mantissas, infinities and NaN among them
    bits = torch.arange(512, dtype=torch.int32)[:, None] * 128 + torch.tensor([0, 1, 37, 64, 127], dtype=torch.int32)
    z = bits.flatten().to(torch.int16).view(torch.bfloat16)
    n = -(-z.numel() // channels) * channels
    values = torch.zeros(-(-n // 64) * 64)
    values[:z.numel()] = z.float()
    values = values.cuda()
    (y0, z0), (y1, z1) = activations(64, values), activations(channels, values[:n])
    y0, z0, y1, z1 = (t[:z.numel()] for t in (y0, z0, y1, z1))
    assert bool(torch.isinf(z0).any() and torch.isnan(z0).any())
    assert torch.equal(torch.isnan(z0), torch.isnan(z1)) and torch.equal(torch.isnan(y0), torch.isnan(y1))
    ok = ~torch.isnan(z0)
    assert torch.equal(z0[ok].view(torch.int16), z1[ok].view(torch.int16))
    ok = ~torch.isnan(y0) & ~(z.abs() < 2.0**-120)
    assert torch.equal(y0[ok].view(torch.int16), y1[ok].view(torch.int16))


@pytest.mark.parametrize("K,O,P", [(24, 160, 840008), (64, 200, 671112), (73, 256, 524296), (40, 320, 420008), (24, 384, 349568)])
def test_long_layers_take_the_formula(lib_built, K, O, P):
    """Few input channels in front of outputs far beyond the caches: the formula in place of the table, the same activations as the shorter pieces give."""
    from makani_amd import pointwise as pw
    from makani_amd._lib import check, lib

    print(f"case gelu formula {K} -> {O}, {P} pixels", flush=True)
    assert 4 * O * P >= 512 << 20
    gen = torch.Generator(device="cuda").manual_seed(K)
    x = torch.randn(K, P, device="cuda", generator=gen).bfloat16()
    w, bias = torch.randn(O, K, device="cuda", generator=gen) / K**0.5, torch.randn(O, device="cuda", generator=gen)
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())

    def conv(x):
        y, z = (torch.empty(O, x.shape[1], dtype=torch.bfloat16, device="cuda") for _ in range(2))
        check(lib.sfno_pointwise_conv_gelu(ptr(x), ptr(pw.packed_weight(w)), ptr(bias), ptr(y), ptr(z), 1, K, O, x.shape[1], pw._stream(x.device)), "forward")
        return y, z

    y, z = conv(x)
    for p in (0, P // 16 * 8, P - 4104):
        ys, zs = conv(x[:, p:p + 4104].contiguous())
        assert torch.equal(y[:, p:p + 4104], ys) and torch.equal(z[:, p:p + 4104], zs)
