"""Weight and bias of the merged layer w (scale x1 + shift) + ws x2 + bias: the stream against packing the composed matrix, bit for bit, the bias against float64."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("O,K,B", [(97, 1, 1), (98, 63, 3), (129, 65, 2), (104, 104, 1), (384, 384, 2), (3, 5, 300)])
@pytest.mark.parametrize("norm,with_bias", [(True, True), (True, False), (False, True)])
def test_merged_weight(lib_built, O, K, B, norm, with_bias):
    from makani_amd import pointwise as pw

    print(f"case merged weight O={O} K={K} B={B} norm={norm} bias={with_bias}", flush=True)
    gen = torch.Generator().manual_seed(O * K + B)
    w, ws = (torch.randn(O, K, generator=gen).cuda() for _ in range(2))
    scale, shift = (torch.randn(B, K, generator=gen).cuda() if norm else None for _ in range(2))
    bias = torch.randn(O, generator=gen).cuda() if with_bias else None
    packed, shifted = pw.merged_weight(w, ws, scale, shift, bias, B)
    torch.cuda.synchronize()
    sh = torch.zeros(B, K, dtype=torch.float64) if shift is None else shift.cpu().double()
    terms = sh[:, None, :] * w.cpu().double()
    ref, size = terms.sum(-1), terms.abs().sum(-1)
    if with_bias:
        ref, size = ref + bias.cpu().double(), size + bias.cpu().double().abs()
    # a chain of ceil(K / 64) products and sums, six foldings, the bias
    assert bool(((shifted.cpu().double() - ref).abs() <= (-(-K // 64) + 7) * 2.0**-24 * size).all())
    for b in range(B):
        left = w if scale is None else w * scale[b]
        assert torch.equal(packed[b], pw.packed_weight(torch.cat([left, ws], dim=1)))


def test_transposed_decoder_weight(lib_built):
    """A network whose decoder weight is a transpose in memory (tied to an encoder's, or taken over with assign=True) gives what its contiguous copy gives."""
    import makani_amd as ma

    print("case merged network, transposed decoder weight", flush=True)
    torch.manual_seed(3)
    net = ma.SphericalFourierNeuralOperatorNet(inp_shape=(48, 96), out_shape=(48, 96), inp_chans=5, out_chans=5, scale_factor=3, embed_dim=104, num_layers=3).cuda().eval()
    x = torch.randn(2, 5, 48, 96, device="cuda")

    def run():
        with torch.inference_mode(), torch.autocast("cuda", dtype=torch.bfloat16):
            return net(x)

    want = run()
    assert net._merge_cache is not None
    conv = net.decoder.fwd[0]
    w = conv.weight.detach().reshape(104, 104)
    conv.weight = torch.nn.Parameter(w.t().contiguous().t()[..., None, None])
    assert not conv.weight.is_contiguous() and torch.equal(conv.weight.detach().reshape(104, 104), w)
    assert torch.equal(run(), want)
    net.merge_decoder = False
    assert float((run().float() - want.float()).norm() / want.float().norm()) < 3e-2


def test_merged_operands(lib_built):
    """Strided operands are read as their values; what does not fit is refused before a kernel reads it."""
    from makani_amd import pointwise as pw

    print("case merged operands", flush=True)
    O, K, B = 104, 40, 3
    gen = torch.Generator().manual_seed(9)
    w, ws, scale, shift, bias = (torch.randn(*s, generator=gen).cuda() for s in ((O, K), (O, K), (B, K), (B, K), (O,)))

    def strided(t):
        return t.t().contiguous().t() if t.dim() == 2 else torch.stack([t, t], 1)[:, 0]

    want = pw.merged_weight(w, ws, scale, shift, bias, B)
    for i in range(5):
        ops = [strided(t) if j == i else t for j, t in enumerate((w, ws, scale, shift, bias))]
        assert not ops[i].is_contiguous()
        assert all(torch.equal(a, b) for a, b in zip(pw.merged_weight(*ops, B), want))
    assert all(torch.equal(a, b) for a, b in zip(pw.merged_weight(w.double(), ws, scale, shift, bias, B), want))
    for bad in ((w.cpu(), ws.cpu(), None, None, None), (w, ws[:, :-1], scale, shift, bias), (w, ws[:-1], scale, shift, bias), (w, ws, scale[:, :-1], shift, bias),
                (w, ws, scale, shift[:-1], bias), (w, ws, scale, None, bias), (w, ws, scale, shift, bias[:-1]), (w, ws, scale, shift, bias.cpu())):
        with pytest.raises(RuntimeError):
            pw.merged_weight(*bad, B)
    x = torch.randn(1, K, 4, 8, generator=gen).bfloat16().cuda()
    stream = want[0][0]
    assert pw.conv1x1_cat(x, x, (O, 2 * K), packed=stream).shape == (1, O, 4, 8)
    for bad in (stream[:-512], stream.float(), stream.cpu(), torch.stack([stream, stream], 1)[:, 0]):
        with pytest.raises(RuntimeError):
            pw.conv1x1_cat(x, x, (O, 2 * K), packed=bad)


def test_skip_of_another_width_is_not_merged(lib_built):
    """A last block whose skip convolution takes more channels than it gives keeps the layer-by-layer tail."""
    import makani_amd as ma

    print("case skip of another width", flush=True)
    torch.manual_seed(4)
    net = ma.SphericalFourierNeuralOperatorNet(inp_shape=(24, 48), out_shape=(24, 48), inp_chans=3, out_chans=3, scale_factor=1, embed_dim=104, num_layers=3).cuda().eval()
    assert net._decoder_merge_ok()
    net.blocks[-1].outer_skip = torch.nn.Conv2d(120, 104, 1, bias=False).cuda()
    assert not net._decoder_merge_ok()
