"""Gradients of the 1x1 convolution on the HIP kernels (bf16 activations) against float64 autograd of the reference op
(nn.Conv2d(kernel_size=1) + bias, makani/models/common/layers.py:95-116,160-216) on the same bf16-rounded operands.

weight / bias gradient: bf16 operands are exact inputs, products exact in fp32, fp32 sums -> relative L2 <= 1e-5, per row of
   the weight gradient too (a row whose pixels were dropped or counted twice fails by far more);
input gradient: the forward kernel on the transposed weight, one bf16 rounding at the store -> relative L2 <= 3e-3."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu


def rel_l2(a, b):
    a, b = a.detach().cpu().double(), b.detach().cpu().double()
    return float(torch.linalg.norm((a - b).ravel()) / max(float(torch.linalg.norm(b.ravel())), 1e-300))


WGRAD_CASES = [
    # B, K, O, H, W, bias
    (1, 20, 36, 13, 8, True),          # one tile, one share, rows and columns far inside the tile
    (2, 73, 384, 20, 36, True),        # encoder: three row tiles, bias column inside the first column tile
    (1, 384, 73, 45, 80, False),       # decoder: two column tiles, the second half empty
    (3, 256, 128, 9, 8, True),         # K = tile width: the bias column opens a second column tile of its own
    (2, 300, 260, 11, 24, True),       # nothing a multiple of the tile sizes; pixels per sample not a multiple of the 32-pixel chunk
    (1, 1, 1, 1, 8, True),             # smallest shape
    (1, 384, 768, 120, 240, True),     # MLP fc1 at a quarter of the model's grid: many shares
    (2, 768, 384, 60, 124, False),     # MLP fc2, two samples, 232.5 chunks per sample
    (1, 257, 70, 24, 16, True),        # one column in the second column tile: the bias belongs to the first only
    (2, 73, 73, 64, 96, False),        # an odd number of entries, 48 shares: the reduction's single loads
    (1, 256, 256, 16, 40, True),       # 65792 entries: its 16-byte loads, few shares (fewer than its wavefronts)
    # enough pixels for tiles of 384 x 192
    (1, 1, 257, 260, 160, True),       # wavefronts without rows or columns, shares of four chunks
    (3, 192, 384, 240, 241, True),     # one full tile, the last chunk of a sample a part
    (2, 384, 384, 200, 212, False),    # two column tiles
    (1, 320, 640, 161, 256, True),     # two row tiles and two column tiles, neither full
    (1, 768, 384, 241, 480, True),     # shares of many chunks
    # and of 192 x 384
    (1, 257, 1, 260, 160, True),
    (3, 384, 192, 240, 241, True),
    (1, 384, 73, 241, 480, True),
]


@pytest.mark.parametrize("B,K,O,H,W,bias", WGRAD_CASES)
def test_weight_and_bias_gradient(lib_built, B, K, O, H, W, bias):
    from makani_amd import pointwise as pw

    assert (H * W) % 8 == 0              # the kernels take H*W a multiple of 8
    print(f"case pointwise wgrad B={B} K={K} O={O} {H}x{W} bias={bias}", flush=True)
    g = torch.Generator().manual_seed(31)
    x = torch.randn(B, K, H, W, generator=g).bfloat16()
    gy = (torch.randn(B, O, H, W, generator=g) * torch.exp(torch.randn(B, O, 1, 1, generator=g))).bfloat16()
    want_w = torch.einsum("bop,bkp->ok", gy.double().reshape(B, O, -1), x.double().reshape(B, K, -1))
    want_b = gy.double().sum(dim=(0, 2, 3))

    gw, gb = pw.conv1x1_weight_grad(gy.cuda(), x.cuda(), bias)
    torch.cuda.synchronize()
    assert gw.shape == (O, K) and gw.dtype == torch.float32
    assert torch.isfinite(gw).all()
    assert rel_l2(gw, want_w) < 1e-5
    rows = torch.linalg.norm(gw.cpu().double() - want_w, dim=1) / torch.linalg.norm(want_w, dim=1).clamp_min(1e-300)
    assert float(rows.max()) < 1e-4, (int(rows.argmax()), float(rows.max()))
    if bias:
        assert gb.shape == (O,) and rel_l2(gb, want_b) < 1e-5
    else:
        assert gb is None
    # the sums run in a fixed order: a second call gives the same bits
    gw2, gb2 = pw.conv1x1_weight_grad(gy.cuda(), x.cuda(), bias)
    torch.cuda.synchronize()
    assert torch.equal(gw, gw2) and (gb is None or torch.equal(gb, gb2))


def test_weight_gradient_counts_every_pixel_once(lib_built):
    """x = 1 and gy = 1 in bf16: every entry of the weight gradient is the number of pixels, exactly, for pixel counts around the
    chunk (32) and share boundaries and for several samples."""
    from makani_amd import pointwise as pw

    for B, P in [(1, 8), (1, 40), (2, 264), (3, 1000), (1, 32 * 4097 + 8)]:
        print(f"case pointwise wgrad count B={B} P={P}", flush=True)
        x = torch.ones(B, 5, 1, P, dtype=torch.bfloat16, device="cuda")
        gy = torch.ones(B, 3, 1, P, dtype=torch.bfloat16, device="cuda")
        gw, gb = pw.conv1x1_weight_grad(gy, x, True)
        torch.cuda.synchronize()
        assert torch.equal(gw.cpu(), torch.full((3, 5), float(B * P))) and torch.equal(gb.cpu(), torch.full((3,), float(B * P)))


@pytest.mark.parametrize("B,K,O,P", [(1, 3, 5, 2 ** 23 + 8), (2, 9, 2, 2 ** 23 + 72), (1, 2, 384, 2 ** 22 - 8), (1, 2, 384, 2 ** 22 + 8)])
def test_rows_too_long_for_32_bit_offsets(lib_built, B, K, O, P):
    """From 2^23 pixels on 256 rows, from 2^22 on 384, lie further apart than 32 bits reach: addresses in 64 bits.  fp32 sums of 1.7e7 products in shares:
    1e-5, as above."""
    from makani_amd import pointwise as pw

    print(f"case pointwise wgrad long rows B={B} P={P}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(7)
    x, gy = (torch.randn(B, c, 8, P // 8, device="cuda", generator=gen).bfloat16() for c in (K, O))
    gw, gb = pw.conv1x1_weight_grad(gy, x, True)
    for o in range(O):
        go = gy[:, o].double()
        want = torch.stack([(go * x[:, k].double()).sum() for k in range(K)])
        # the sums of independent products cancel to sqrt(B P); relative to that
        assert float((gw[o].double() - want).abs().max()) < 1e-5 * (B * P) ** 0.5
        assert float((gb[o].double() - go.sum()).abs()) < 1e-5 * (B * P) ** 0.5


AUTOGRAD_CASES = [
    # B, K, O, H, W, bias, x requires grad
    (2, 73, 384, 20, 36, True, False),      # first layer of the encoder: the input needs no gradient
    (1, 384, 768, 16, 24, True, True),
    (2, 768, 384, 13, 8, False, True),
    (1, 100, 200, 11, 24, True, True),
]


@pytest.mark.parametrize("B,K,O,H,W,bias,xgrad", AUTOGRAD_CASES)
def test_trainable_convolution_against_float64_autograd(lib_built, B, K, O, H, W, bias, xgrad):
    from makani_amd import pointwise as pw

    print(f"case pointwise autograd B={B} K={K} O={O} {H}x{W} bias={bias} xgrad={xgrad}", flush=True)
    g = torch.Generator().manual_seed(41)
    x = torch.randn(B, K, H, W, generator=g).bfloat16()
    w = torch.randn(O, K, 1, 1, generator=g) / np.sqrt(K)
    bvec = torch.randn(O, generator=g) if bias else None
    gy = torch.randn(B, O, H, W, generator=g).bfloat16()

    # float64 reference on the operands as the kernels see them (bf16 activations, bf16-rounded weight)
    xr = x.double().requires_grad_(xgrad)
    wr = w.bfloat16().double().requires_grad_(True)
    br = bvec.double().requires_grad_(True) if bias else None
    F.conv2d(xr, wr, br).backward(gy.double())

    conv = pw.PointwiseConv2d(K, O, bias=bias).cuda()
    with torch.no_grad():
        conv.weight.copy_(w)
        if bias:
            conv.bias.copy_(bvec)
    xg = x.cuda().requires_grad_(xgrad)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = conv(xg)
    assert y.dtype == torch.bfloat16 and y.grad_fn is not None and type(y.grad_fn).__name__.startswith("_Conv1x1")
    y.backward(gy.cuda())
    torch.cuda.synchronize()
    assert rel_l2(y, F.conv2d(x.double(), w.bfloat16().double(), bvec.double() if bias else None)) < 3e-3
    assert conv.weight.grad.dtype == torch.float32 and conv.weight.grad.shape == w.shape
    assert rel_l2(conv.weight.grad, wr.grad) < 1e-5
    if bias:
        assert rel_l2(conv.bias.grad, br.grad) < 1e-5
    if xgrad:
        assert xg.grad.dtype == torch.bfloat16 and rel_l2(xg.grad, xr.grad) < 3e-3
    else:
        assert xg.grad is None


def test_pointwise_conv2d_is_nn_conv2d_elsewhere(lib_built):
    """Without a gradient, in fp32 or on the CPU the module is nn.Conv2d: same values, same state-dict keys."""
    from makani_amd import pointwise as pw

    print("case pointwise module fallback", flush=True)
    torch.manual_seed(5)
    conv = pw.PointwiseConv2d(12, 7, bias=True)
    ref = torch.nn.Conv2d(12, 7, 1, bias=True)
    assert list(conv.state_dict().keys()) == list(ref.state_dict().keys())
    ref.load_state_dict(conv.state_dict())
    x = torch.randn(2, 12, 4, 8)
    assert torch.equal(conv(x), ref(x))                                   # CPU
    conv, ref, x = conv.cuda(), ref.cuda(), x.cuda()
    y = conv(x.requires_grad_(True))                                      # fp32 with a gradient: the library's convolution
    assert y.dtype == torch.float32 and not type(y.grad_fn).__name__.startswith("_Conv1x1")
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        assert torch.equal(conv(x), ref(x))                               # bf16 without a gradient


def test_training_step_through_the_network_matches_the_module_path(lib_built):
    """One forward + backward of a small SFNO under bf16 autocast in training mode: the 1x1 convolutions run on the HIP kernels
    in both directions (their nodes are in the graph) and every parameter gradient agrees with the same network evaluated with
    nn.Conv2d's own kernels to bf16 accuracy."""
    import makani_amd as ma
    from makani_amd import pointwise as pw

    print("case pointwise training step", flush=True)
    torch.manual_seed(11)
    kw = dict(inp_shape=(33, 64), out_shape=(33, 64), inp_chans=5, out_chans=3, scale_factor=2, embed_dim=32, num_layers=2)
    net = ma.SphericalFourierNeuralOperatorNet(**kw).cuda().train()
    x = torch.randn(2, 5, 33, 64, device="cuda")
    tgt = torch.randn(2, 3, 33, 64, device="cuda")

    def grads(use_hip):
        net.zero_grad(set_to_none=True)
        saved = pw.trainable_active
        if not use_hip:
            pw.trainable_active = lambda t: False
        try:
            with torch.autocast("cuda", dtype=torch.bfloat16):
                y = net(x)
            names = set()
            stack = [y.grad_fn]
            seen = set()
            while stack:
                f = stack.pop()
                if f is None or f in seen:
                    continue
                seen.add(f)
                names.add(type(f).__name__)
                stack.extend(n for n, _ in f.next_functions)
            loss = ((y.float() - tgt) ** 2).mean()
            loss.backward()
        finally:
            pw.trainable_active = saved
        torch.cuda.synchronize()
        real = lambda t: torch.view_as_real(t) if t.is_complex() else t
        return float(loss.detach()), {n: real(p.grad.detach()).clone() for n, p in net.named_parameters() if p.grad is not None}, names

    l_hip, g_hip, names_hip = grads(True)
    l_ref, g_ref, names_ref = grads(False)
    assert any(n.startswith("_Conv1x1") for n in names_hip) and not any(n.startswith("_Conv1x1") for n in names_ref)
    assert abs(l_hip - l_ref) <= 2e-2 * abs(l_ref)
    assert set(g_hip) == set(g_ref) and len(g_hip) > 10
    # (a bias in front of an instance norm has a zero gradient up to rounding noise: parameters whose gradient is far below the
    # largest one are judged together with the others, not one by one)
    norms = {n: float(torch.linalg.norm(g_ref[n].double())) for n in g_ref}
    top = max(norms.values())
    worst = max((rel_l2(g_hip[n], g_ref[n]), n) for n in g_ref if norms[n] > 1e-2 * top)
    assert worst[0] < 5e-2, worst
    err = sum(float(torch.linalg.norm((g_hip[n] - g_ref[n]).double())) ** 2 for n in g_ref) ** 0.5
    assert err < 3e-2 * sum(v * v for v in norms.values()) ** 0.5


@pytest.mark.parametrize("channels", [8, 104])
def test_training_gelu_and_its_derivative_on_every_bf16_value(lib_built, channels):
    """conv -> GELU and the GELU's derivative in the convolutions' epilogues, through an identity matrix, at every bf16 value between -6
    and 8.  fp32 arithmetic (2^-23 of Phi) and one rounding to bf16: half a unit of the result and 3e-7 beside it.  An activation within
    the fp32 error (1e-6 relative in the tail) of a rounding boundary may fall on its other side: 2e-6 / 2^-8, one of the 2242 values
    from 2^-6 on."""
    import ctypes

    from makani_amd import pointwise as pw
    from makani_amd._lib import check, lib

    print(f"case training gelu {channels}", flush=True)
    z = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16)
    z = z[torch.isfinite(z) & (z >= -6) & (z <= 8)]
    P = (z.numel() // channels + 8) // 8 * 8
    x = torch.zeros(channels * P, dtype=torch.bfloat16)
    x[:z.numel()] = z
    x = x.reshape(1, channels, 1, P).cuda()
    eye, ones = torch.eye(channels, device="cuda"), torch.ones_like(x)
    y, pre, gx = (torch.empty_like(x) for _ in range(3))
    ptr = lambda t: ctypes.c_void_p(t.data_ptr())
    check(lib.sfno_pointwise_conv_gelu(ptr(x), ptr(pw.packed_weight(eye)), None, ptr(y), ptr(pre), 1, channels, channels, P, pw._stream(x.device)), "forward")
    check(lib.sfno_pointwise_conv_gelu_grad(ptr(ones), ptr(pw.packed_weight(eye, transposed=True)), ptr(x), ptr(gx), 1, channels, channels, P,
                                            pw._stream(x.device)), "backward")
    torch.cuda.synchronize()
    xd = x.double().cpu()
    assert torch.equal(pre.float().cpu(), x.float().cpu())
    Phi = 0.5 * torch.special.erfc(-xd / 2 ** 0.5)
    pdf = torch.exp(-0.5 * xd * xd) / (2 * torch.pi) ** 0.5
    want = xd * Phi
    got = y.double().cpu()
    assert bool(((got - want).abs() <= want.abs() * 2 ** -8 + 3e-7).all())
    assert int(((got != want.to(torch.bfloat16).double()) & (xd.abs() >= 2 ** -6)).sum()) < 5
    want = Phi + xd * pdf
    assert bool(((gx.double().cpu() - want).abs() <= want.abs() * 2 ** -8 + 3e-7).all())


def test_views_between_16_byte_boundaries(lib_built):
    """Tensors that start in the middle of a buffer give the results of their copies, in every function that takes activations."""
    import torch.nn as nn

    from makani_amd import pointwise as pw
    from makani_amd.sfnonet import EncoderDecoder

    print("case offsets", flush=True)
    torch.manual_seed(3)

    def offset(t):
        return torch.cat([t.new_zeros(3), t.flatten()])[3:].view(t.shape)

    x, r = (torch.randn(2, 12, 8, 16, device="cuda").bfloat16() for _ in range(2))
    w, sc, sh = torch.randn(12, 12, device="cuda"), torch.randn(2, 12, device="cuda"), torch.randn(2, 12, device="cuda")
    wcat = torch.randn(100, 24, device="cuda")
    calls = [lambda x, r: pw.conv1x1(x, w, None, "gelu", r, sc, sh), lambda x, r: pw.conv1x1_cat(x, r, wcat), lambda x, r: torch.stack(pw.instance_norm_coeffs(x)),
             lambda x, r: pw.scale_shift_act(x, sc, sh, "gelu"), lambda x, r: pw.conv1x1_weight_grad(r, x, True)[0]]
    for i, f in enumerate(calls):
        assert torch.equal(f(offset(x), offset(r)), f(x, r)), i
    for mod in (EncoderDecoder(1, 12, 12, 20, nn.GELU).cuda(), pw.PointwiseConv2d(12, 12).cuda()):
        got = []
        for view in (offset, torch.clone):
            xi = view(x).requires_grad_()
            with torch.autocast("cuda", dtype=torch.bfloat16):
                y = mod(xi)
            got.append((y, *torch.autograd.grad(y, (xi, *mod.parameters()), view(r))))
        assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("transposed", [False, True])
def test_packed_weight_on_another_stream(lib_built, transposed):
    """A weight packed behind other work of one stream is used by the next stream at once: that stream waits for the packing."""
    from makani_amd import pointwise as pw

    print("case packed weight, two streams", transposed, flush=True)
    torch.manual_seed(4)
    w, x = torch.randn(24, 24, device="cuda"), torch.randn(1, 24, 16, 16, device="cuda").bfloat16()
    pw._conv1x1(x, w, transposed)
    pw.clear_cache(w)
    a, b = torch.cuda.Stream(), torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(a):
        torch.cuda._sleep(20_000_000)
        p = pw.packed_weight(w, transposed)
    with torch.cuda.stream(b):
        got = pw._conv1x1(x, w, transposed)
        again = pw._conv1x1(x, w, transposed)
    assert pw.packed_weight(w, transposed) is p
    torch.cuda.synchronize()
    pw.clear_cache(w)
    want = pw._conv1x1(x, w, transposed)
    assert torch.equal(got, want) and torch.equal(again, want)


@pytest.mark.parametrize("O,K", [(1, 1), (73, 384), (384, 73), (97, 128), (130, 260), (31, 64)])
def test_weight_and_transpose_packed_together(lib_built, O, K):
    """One launch writes what the two separate packings write, padding included."""
    from makani_amd import pointwise as pw

    w = torch.randn(O, K, 1, 1, generator=torch.Generator().manual_seed(8)).cuda()
    want = [pw.packed_weight(w, transposed=t).clone() for t in (False, True)]
    pw.clear_cache(w)
    p = pw.packed_weight(w, both=True)
    hit = [pw._wcache[(id(w), t)][2] for t in (False, True)]
    assert hit[0] is p and pw.packed_weight(w, transposed=True) is hit[1]
    assert torch.equal(hit[0], want[0]) and torch.equal(hit[1], want[1])
