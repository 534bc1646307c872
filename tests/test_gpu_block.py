"""The native block (makani_amd/block.py, csrc/block.cpp) and the convolution -> GELU -> convolution pair of encoder and decoder in
training: output and every gradient against the same modules in float32, next to the layer-by-layer modules under bf16 autocast.

Bound: both bf16 evaluations round the output of a layer to 8 bits (2^-8 / sqrt 3 / 1.4 = 1.7e-3 relative L2 each).  About a dozen such
roundings lie between an input and a gradient, sqrt(12) 1.7e-3 = 6e-3, up to twice that where a norm or a cancelling sum amplifies
them: 1.5e-2 asserted.  The native block rounds less often than the modules, so its error may exceed theirs by sampling only (a
quarter, plus 1e-3)."""
import contextlib

import pytest
import torch
import torch.nn as nn

pytestmark = pytest.mark.gpu


def rel(a, b):
    a, b = (torch.view_as_real(t) if t.is_complex() else t for t in (a.detach(), b.detach()))
    return float((a.double() - b.double()).norm() / b.double().norm().clamp_min(1e-300))


def make_block(fwd, inv, embed, ratio, affine=True):
    from functools import partial

    from makani_amd.sfnonet import FourierNeuralOperatorBlock

    norm = partial(nn.InstanceNorm2d, num_features=embed, eps=1e-6, affine=affine, track_running_stats=False)
    blk = FourierNeuralOperatorBlock(fwd, inv, embed, operator_type="dhconv", mlp_ratio=ratio, norm_layer=(norm, norm), inner_skip="none", outer_skip="linear",
                                     use_mlp=True)
    with torch.no_grad():
        for p in blk.parameters():
            if not p.is_complex() and p.dim() == 1:
                p.add_(0.2 * torch.randn(p.shape))
    return blk.cuda()


def passes(blk, x, gy, autocast, leaf=None):
    for p in blk.parameters():
        p.grad = None
    xi = x.clone().requires_grad_()
    with torch.autocast("cuda", dtype=torch.bfloat16) if autocast else contextlib.nullcontext():
        y = blk(xi)
    y.backward(gy.to(y.dtype))
    return {"y": y, "x": xi.grad, **{n: p.grad.clone() for n, p in blk.named_parameters()}}


CASES = [
    # forward grid, inverse grid, batch, embed, MLP ratio
    ((32, 64, "legendre-gauss"), (32, 64, "legendre-gauss"), 2, 24, 2.0),       # equal grids: the residual is the input
    ((33, 64, "equiangular"), (16, 32, "legendre-gauss"), 3, 36, 1.5),          # down: the residual goes through the transforms, padded channel slots
    ((16, 32, "legendre-gauss"), (33, 64, "equiangular"), 1, 104, 2.0),         # up
    ((24, 48, "planar"), (24, 48, "planar"), 2, 17, 3.0),                       # planar pair, odd channels
]


@pytest.mark.parametrize("f,i,B,E,ratio", CASES)
def test_block_gradients(lib_built, f, i, B, E, ratio):
    import makani_amd as ma
    from makani_amd import block as nb

    print(f"case block {f} -> {i} B={B} E={E}", flush=True)
    torch.manual_seed(4)
    lmax, mmax = min(f[0], i[0]) - (i[2] == "planar") * 3, min(f[1], i[1]) // 2 + 1
    if f[2] == "planar":
        fwd, inv = ma.RealFFT2(*f[:2], lmax, mmax), ma.InverseRealFFT2(*i[:2], lmax, mmax)
    else:
        fwd, inv = ma.RealSHT(*f[:2], lmax=lmax, mmax=mmax, grid=f[2]), ma.InverseRealSHT(*i[:2], lmax=lmax, mmax=mmax, grid=i[2])
    blk = make_block(fwd, inv, E, ratio, affine=B != 3)
    x = torch.randn(B, E, *f[:2], device="cuda").to(torch.bfloat16)
    gy = torch.randn(B, E, *i[:2], device="cuda").to(torch.bfloat16)
    calls = []
    keep = nb._BlockFn.apply
    nb._BlockFn.apply = lambda *a: calls.append(1) or keep(*a)
    try:
        got = passes(blk, x, gy, True)
    finally:
        nb._BlockFn.apply = keep
    assert calls
    again = passes(blk, x, gy, True)
    blk.fused_pointwise = False
    mod = passes(blk, x, gy, True)
    ref = passes(blk, x.float(), gy.float(), False)
    for n, r in ref.items():
        if n == "mlp.fwd.3.bias":
            continue                      # in front of an instance norm: its gradient is zero but for rounding
        assert torch.equal(got[n], again[n]), n
        e, em = rel(got[n], r), rel(mod[n], r)
        assert e < 1.5e-2 and e < 1.25 * em + 1e-3, (n, e, em)
    # inference: the same block without a gradient
    blk.fused_pointwise = True
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        assert rel(blk.eval()(x), ref["y"]) < 1.5e-2


@pytest.mark.parametrize("grid,B,E", [((4, 8), 4, 32), ((16, 32), 1, 5), ((9, 24), 2, 3), ((64, 64), 1, 4)])
def test_norm_of_a_small_grid_follows_the_stored_field(lib_built, grid, B, E):
    """Up to 4096 pixels norm0 takes the moments of the field as it is stored: with those of the field before its rounding to bf16 the
    normalised field keeps the mean of the rounding errors (2^-9 / sqrt(3 P) of the field: 2e-4 at 32 pixels).  Moments in fp32 from
    exact values: 1e-6 of the standard deviation asserted."""
    import makani_amd as ma
    from makani_amd import block as nb

    print(f"case small norm {grid} B={B} E={E}", flush=True)
    torch.manual_seed(9)
    fwd, inv = ma.RealSHT(*grid, grid="legendre-gauss"), ma.InverseRealSHT(*grid, grid="legendre-gauss")
    blk = make_block(fwd, inv, E, 2.0)
    x = (3.0 + torch.randn(B, E, *grid, device="cuda")).to(torch.bfloat16)
    c = nb._Call(blk, x, nb.block_params(blk))
    kept = c.forward(x, 1, torch.empty_like(x))
    rows, P = B * E, grid[0] * grid[1]

    def part(i, n, dtype):
        return kept[c.offsets[i]:c.offsets[i] + n * dtype.itemsize].view(dtype)

    xf = part(1, rows * P, torch.bfloat16).view(rows, P).double()
    mean, rstd = part(2, 4 * rows, torch.float32)[2 * rows:].view(rows, 2).double().unbind(1)
    want = 1.0 / (xf.var(1, unbiased=False) + blk.norm0.eps).sqrt()
    assert float(((mean - xf.mean(1)).abs() * want).max()) < 1e-6
    assert float((rstd / want - 1.0).abs().max()) < 1e-6
    # the module path on these grids too
    assert not blk._norm0_from_transform()


def test_frozen_parameters_and_input(lib_built):
    """Only what asks for a gradient gets one."""
    import makani_amd as ma

    torch.manual_seed(5)
    sht, isht = ma.RealSHT(16, 32, grid="legendre-gauss"), ma.InverseRealSHT(16, 32, grid="legendre-gauss")
    blk = make_block(sht, isht, 16, 2.0)
    x = torch.randn(1, 16, 16, 32, device="cuda").to(torch.bfloat16)
    names = [n for n, _ in blk.named_parameters()]
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = blk(x)
        full = dict(zip(names, torch.autograd.grad(y.float().square().sum(), list(blk.parameters()))))
    for only in names:
        if only == "mlp.fwd.3.bias":
            continue
        for n, p in blk.named_parameters():
            p.requires_grad_(n == only)
            p.grad = None
        with torch.autocast("cuda", dtype=torch.bfloat16):
            blk(x).float().square().sum().backward()
        for n, p in blk.named_parameters():
            assert (p.grad is not None) == (n == only), n
            if n == only:
                assert torch.equal(p.grad, full[n]), n


def test_backward_uses_the_values_of_the_forward(lib_built):
    """A functional call swaps other values in for the forward only; a strided parameter is read as its values, not as its memory."""
    import makani_amd as ma

    torch.manual_seed(6)
    sht, isht = ma.RealSHT(16, 32, grid="legendre-gauss"), ma.InverseRealSHT(16, 32, grid="legendre-gauss")
    a, b = make_block(sht, isht, 16, 2.0), make_block(sht, isht, 16, 2.0)
    x = torch.randn(1, 16, 16, 32, device="cuda").to(torch.bfloat16)
    want = passes(b, x, torch.ones_like(x), True)
    values = {}
    for n, p in b.named_parameters():
        store = torch.empty(*p.shape, 2, dtype=p.dtype, device=p.device)
        store[..., 0] = p.detach()
        values[n] = store[..., 0].requires_grad_()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = torch.func.functional_call(a, values, (x,))
    grads = torch.autograd.grad(y, list(values.values()), torch.ones_like(y))
    assert torch.equal(y, want["y"])
    for n, g in zip(values, grads):
        assert torch.equal(g, want[n]), n


def test_subclassed_convolutions_and_global_hooks_keep_the_modules(lib_built):
    import makani_amd as ma

    class Doubled(nn.Conv2d):
        def forward(self, x):
            return 2.0 * super().forward(x)

    torch.manual_seed(7)
    sht, isht = ma.RealSHT(16, 32, grid="legendre-gauss"), ma.InverseRealSHT(16, 32, grid="legendre-gauss")
    blk = make_block(sht, isht, 16, 2.0)
    x = torch.randn(1, 16, 16, 32, device="cuda").to(torch.bfloat16)
    gy = torch.randn_like(x)
    seen = []
    handle = nn.modules.module.register_module_forward_hook(lambda m, a, y: seen.append(m))
    try:
        passes(blk, x, gy, True)
    finally:
        handle.remove()
    assert blk.mlp.fwd[0] in seen and blk.norm1 in seen
    fc1 = Doubled(16, 32, 1).cuda()
    fc1.load_state_dict(blk.mlp.fwd[0].state_dict())
    blk.mlp.fwd[0] = fc1
    ref = passes(blk, x.float(), gy.float(), False)
    assert rel(passes(blk, x, gy, True)["y"], ref["y"]) < 1.5e-2


@pytest.mark.parametrize("cin,hid,cout,H,W", [(5, 33, 7, 12, 16), (73, 128, 100, 24, 32), (16, 200, 130, 40, 64)])
def test_conv_gelu_conv(lib_built, cin, hid, cout, H, W):
    from makani_amd.sfnonet import EncoderDecoder

    print(f"case chain {cin} {hid} {cout}", flush=True)
    torch.manual_seed(6)
    enc = EncoderDecoder(1, cin, cout, hid, nn.GELU).cuda()
    with torch.no_grad():
        enc.fwd[0].bias.normal_()
    x = torch.randn(2, cin, H, W, device="cuda")
    gy = torch.randn(2, cout, H, W, device="cuda")
    got = passes(enc, x, gy, True)
    ref = passes(enc, x, gy, False)
    for n, r in ref.items():
        assert rel(got[n], r) < 1e-2, n


def test_conv_gelu_conv_refuses_other_channel_counts(lib_built):
    """The packed weights are addressed by the input's channel count: a wrong one is an error of the host, not a read past them."""
    from makani_amd.sfnonet import EncoderDecoder

    enc = EncoderDecoder(1, 6, 5, 8, nn.GELU).cuda()
    for channels in (5, 7):
        with torch.autocast("cuda", dtype=torch.bfloat16), pytest.raises(RuntimeError):
            enc(torch.randn(1, channels, 8, 16, device="cuda"))
    enc.fwd[2] = nn.Conv2d(9, 5, 1).cuda()
    with torch.autocast("cuda", dtype=torch.bfloat16), pytest.raises(RuntimeError):
        enc(torch.randn(1, 6, 8, 16, device="cuda"))


def test_offset_tensors_and_foreign_shapes(lib_built):
    """Views that start between 16-byte boundaries give the results of their copies; inputs and parameters of another size raise."""
    import makani_amd as ma

    torch.manual_seed(8)
    sht, isht = ma.RealSHT(16, 32, grid="legendre-gauss"), ma.InverseRealSHT(16, 32, grid="legendre-gauss")
    blk = make_block(sht, isht, 16, 2.0)
    x, gy = (torch.randn(1, 16, 16, 32, device="cuda").to(torch.bfloat16) for _ in range(2))

    def offset(t):
        return torch.cat([t.new_zeros(1), t.flatten()])[1:].view(t.shape)

    want = passes(blk, x, gy, True)
    got = passes(blk, x, offset(gy), True)
    for n, w in want.items():
        assert torch.equal(got[n], w), n
    with torch.no_grad(), torch.autocast("cuda", dtype=torch.bfloat16):
        assert rel(blk.eval()(offset(x)), want["y"].float()) < 1.5e-2
    for mode in (torch.enable_grad, torch.no_grad):
        with mode(), torch.autocast("cuda", dtype=torch.bfloat16), pytest.raises(RuntimeError):
            blk(x[:, :15].contiguous())
    blk.mlp.fwd[0] = nn.Conv2d(15, 32, 1).cuda()
    with torch.autocast("cuda", dtype=torch.bfloat16), pytest.raises(RuntimeError):
        blk.train()(x)


@pytest.mark.parametrize("at_construction", [True, False])
def test_switch_reaches_encoder_and_decoder_in_training(lib_built, at_construction, monkeypatch):
    """fused_pointwise=False keeps the modules of encoder and decoder too while gradients are recorded."""
    from makani_amd import block as nb, pointwise as pw
    from makani_amd.sfnonet import SphericalFourierNeuralOperatorNet

    calls = []
    for fn in (pw._ConvGeluConv, nb._BlockFn):
        monkeypatch.setattr(fn, "apply", lambda *a, f=fn, keep=fn.apply: calls.append(f) or keep(*a))
    torch.manual_seed(10)
    net = SphericalFourierNeuralOperatorNet(inp_shape=(33, 64), out_shape=(33, 64), inp_chans=3, out_chans=3, scale_factor=2, embed_dim=16, num_layers=2,
                                            fused_pointwise=not at_construction).cuda()
    x = torch.randn(1, 3, 33, 64, device="cuda")
    with torch.autocast("cuda", dtype=torch.bfloat16):
        if not at_construction:
            net(x)
            assert calls.count(pw._ConvGeluConv) == 2 and calls.count(nb._BlockFn) == 2
            calls.clear()
            net.fused_pointwise = False
            for b in net.blocks:
                b.fused_pointwise = False
        net(x).float().square().sum().backward()
    assert not calls and all(p.grad is not None for p in net.parameters())


def test_kernels_train_only_what_asks_for_a_gradient(lib_built, monkeypatch):
    """With gradients enabled but asked for by nothing, the modules run (as they do for each convolution by itself)."""
    import makani_amd as ma
    from makani_amd import block as nb, pointwise as pw
    from makani_amd.sfnonet import EncoderDecoder

    calls = []
    for fn in (pw._ConvGeluConv, nb._BlockFn):
        monkeypatch.setattr(fn, "apply", lambda *a, f=fn, keep=fn.apply: calls.append(f) or keep(*a))
    torch.manual_seed(11)
    sht, isht = ma.RealSHT(16, 32, grid="legendre-gauss"), ma.InverseRealSHT(16, 32, grid="legendre-gauss")
    blk, enc = make_block(sht, isht, 16, 2.0).requires_grad_(False), EncoderDecoder(1, 16, 16, 16, nn.GELU).cuda().requires_grad_(False)
    x = torch.randn(1, 16, 16, 32, device="cuda").to(torch.bfloat16)
    for mod in (blk, enc):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = mod(x)
            assert not calls and not y.requires_grad
            mod(x.clone().requires_grad_()).float().sum().backward()
            assert len(calls) == 1
            next(mod.parameters()).requires_grad_()
            mod(x).float().sum().backward()
            assert len(calls) == 2
        calls.clear()


def test_library_convolutions_keep_their_second_derivative(lib_built):
    """nn.Conv2d in the place of the package's convolution trains on the library's kernels and can be differentiated twice."""
    from makani_amd.sfnonet import EncoderDecoder

    torch.manual_seed(12)
    enc = EncoderDecoder(1, 6, 5, 8, nn.GELU).cuda()
    for i in (0, 2):
        conv = nn.Conv2d(*enc.fwd[i].weight.shape[1::-1], 1, bias=enc.fwd[i].bias is not None).cuda()
        conv.load_state_dict(enc.fwd[i].state_dict())
        enc.fwd[i] = conv
    x = torch.randn(1, 6, 8, 16, device="cuda", requires_grad=True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        (g,) = torch.autograd.grad(enc(x).float().square().sum(), x, create_graph=True)
    g.square().sum().backward()
    assert all(p.grad is not None and torch.isfinite(p.grad).all() for p in enc.parameters())


def test_backward_refuses_foreign_buffers_plans_and_weights(lib_built):
    """The C entry points check what they address by the block's sizes before anything is enqueued."""
    import ctypes

    import makani_amd as ma
    from makani_amd import _lib, block as nb
    from makani_amd._lib import lib
    from makani_amd.contractions import packed_for

    torch.manual_seed(13)
    sht, isht = ma.RealSHT(16, 32, grid="legendre-gauss"), ma.InverseRealSHT(16, 32, grid="legendre-gauss")
    blk = make_block(sht, isht, 16, 2.0)
    x = torch.randn(1, 16, 16, 32, device="cuda").to(torch.bfloat16)
    out, gx = torch.empty_like(x), torch.empty_like(x)
    EINVAL, EWORKSPACE = -1, -4
    c = nb._Call(blk, x, nb.block_params(blk), backward=True)
    kept = c.forward(x, 1, out)
    grads = _lib.BlockGrads(gx=gx.data_ptr())
    ref = ctypes.byref(c.b)
    nws = lib.sfno_block_workspace_bytes(ref, 1)
    ws = torch.empty(max(nws, lib.sfno_block_workspace_bytes(ref, 0)), dtype=torch.uint8, device="cuda")

    def backward(kept_bytes):
        return lib.sfno_block_backward(ref, x.data_ptr(), x.data_ptr(), kept.data_ptr(), kept_bytes, ctypes.byref(grads), ws.data_ptr(), nws, c.stream)

    assert backward(kept.numel()) == 0
    assert backward(kept.numel() - 1) == EWORKSPACE
    small = lib.sfno_block_layout(ref, 0, c.offsets)
    assert small < kept.numel() and backward(small) == EWORKSPACE
    other = ma.RealSHT(24, 48, grid="legendre-gauss").plan(x.device, adjoint=True), ma.InverseRealSHT(24, 48, grid="legendre-gauss").plan(x.device, adjoint=True)
    weight = torch.randn(16, 8, 16, dtype=torch.complex64, device="cuda")
    for field, value in (("fwd_adj", other[0].handle), ("inv_adj", other[1].handle), ("fwd_adj", c.keep[0].handle), ("inv_adj", None),
                         ("weights_adj", packed_for(weight, adjoint=True).handle), ("weights_adj", None), ("w2t", None), ("wskipt", None)):
        keep = getattr(c.b, field)
        setattr(c.b, field, value)
        assert backward(kept.numel()) == EINVAL, field
        setattr(c.b, field, keep)
    bias = torch.empty(32, device="cuda")
    grads.gb1 = bias.data_ptr()                # a bias without its matrix
    assert backward(kept.numel()) == EINVAL
    keep = c.b.weights
    c.b.weights = packed_for(weight).handle
    assert lib.sfno_block_forward(ref, 1, x.data_ptr(), out.data_ptr(), kept.data_ptr(), kept.numel(), ws.data_ptr(), ws.numel(), c.stream) == EINVAL
    c.b.weights = keep
    torch.cuda.synchronize()


def peak_of(call):
    """Bytes beside what is allocated before and after the call."""
    call()                                            # packed weights, plans
    torch.cuda.synchronize()
    base = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    call()
    torch.cuda.synchronize()
    return torch.cuda.max_memory_allocated() - base


@pytest.mark.parametrize("f,i", [((64, 128), (64, 128)), ((64, 128), (32, 64)), ((32, 64), (64, 128))])
def test_peak_memory_of_inference_is_no_more_than_layer_by_layer(lib_built, f, i, monkeypatch):
    """The call's buffers are laid over each other: what it needs beside its input does not exceed what the layers need one after
    the other (the block may hand its last sum on)."""
    import makani_amd as ma
    from makani_amd import block as nb

    print(f"case peak {f} -> {i}", flush=True)
    torch.manual_seed(14)
    lmax, mmax = min(f[0], i[0]), min(f[1], i[1]) // 2 + 1
    fwd = ma.RealSHT(*f, lmax=lmax, mmax=mmax, grid="legendre-gauss")
    blk = make_block(fwd, ma.InverseRealSHT(*i, lmax=lmax, mmax=mmax, grid="legendre-gauss"), 64, 2.0).eval()
    x = torch.randn(2, 64, *f, device="cuda").to(torch.bfloat16)

    @torch.autocast("cuda", dtype=torch.bfloat16)
    @torch.no_grad()
    def call():
        blk(x, defer_skip=True)

    native = peak_of(call)
    monkeypatch.setattr(nb, "supported", lambda *a: False)
    assert native <= peak_of(call) + (1 << 16)        # rounding of some dozen allocations


def test_peak_memory_of_training_is_that_of_layer_by_layer(lib_built):
    """What a block kept is given back at the end of its backward only, layer by layer it goes piece by piece, but with more tensors on
    their way: a twentieth more at most (at 721 x 1440 it is less)."""
    from makani_amd.sfnonet import SphericalFourierNeuralOperatorNet

    torch.manual_seed(15)
    net = SphericalFourierNeuralOperatorNet(inp_shape=(65, 128), out_shape=(65, 128), inp_chans=6, out_chans=6, scale_factor=2, embed_dim=64, num_layers=4).cuda()
    x = torch.randn(2, 6, 65, 128, device="cuda")

    def call():
        with torch.autocast("cuda", dtype=torch.bfloat16):
            net(x).float().square().mean().backward()
        net.zero_grad(set_to_none=True)

    native = peak_of(call)
    net.fused_pointwise = False
    for b in net.blocks:
        b.fused_pointwise = False
    assert native <= 1.05 * peak_of(call)


def test_blocks_without_a_norm_train_on_the_modules(lib_built):
    from makani_amd.sfnonet import SphericalFourierNeuralOperatorNet

    torch.manual_seed(16)
    net = SphericalFourierNeuralOperatorNet(inp_shape=(33, 64), out_shape=(33, 64), inp_chans=3, out_chans=3, scale_factor=2, embed_dim=16, num_layers=2,
                                            normalization_layer="none").cuda()
    x = torch.randn(1, 3, 33, 64, device="cuda")
    with torch.autocast("cuda", dtype=torch.bfloat16):
        net(x).float().square().mean().backward()
        with torch.no_grad():
            y = net.eval()(x)
    assert torch.isfinite(y).all() and all(p.grad is not None for p in net.parameters())


def test_every_block_of_a_network_is_one_native_call(lib_built):
    """Under autocast the skip weight folded with the encoder stays float32, so the first block is served like the others."""
    import makani_amd as ma
    from makani_amd import block as nb

    torch.manual_seed(8)
    net = ma.SphericalFourierNeuralOperatorNet(inp_shape=(32, 64), out_shape=(32, 64), scale_factor=4, inp_chans=3, out_chans=3, embed_dim=16, num_layers=3,
                                               operator_type="dhconv").cuda().eval()
    x = torch.randn(2, 3, 32, 64, device="cuda")
    calls = []
    keep = nb.forward
    nb.forward = lambda *a, **k: calls.append(1) or keep(*a, **k)
    try:
        with torch.inference_mode(), torch.autocast("cuda", dtype=torch.bfloat16):
            got = net(x)
    finally:
        nb.forward = keep
    assert len(calls) == 3 and net._fold_cache[2].dtype == torch.float32
    net.fused_pointwise = False
    for b in net.blocks:
        b.fused_pointwise = False
    with torch.inference_mode():
        assert rel(got, net(x)) < 3e-2


def test_adjoint_packings_follow_the_backward(lib_built):
    """A forward that records gradients packs no adjoint before a backward has asked for one, a backward without the input's gradient asks for
    those it reads only, and from then on a changed weight and its adjoint are packed together."""
    import makani_amd as ma
    from makani_amd import block as nb
    from makani_amd import contractions as C
    from makani_amd import pointwise as pw

    torch.manual_seed(9)
    fwd, inv = ma.RealSHT(16, 32, grid="legendre-gauss"), ma.InverseRealSHT(16, 32, grid="legendre-gauss")
    blk = make_block(fwd, inv, 24, 2.0)
    x, gy = (torch.randn(2, 24, 16, 32, device="cuda").to(torch.bfloat16) for _ in range(2))
    fc1, fc2 = nb.mlp_convs(blk)
    ws = {"filter": blk.filter.filter.weight, "skip": blk.outer_skip.weight, "fc1": fc1.weight, "fc2": fc2.weight}

    def adjoints():
        return {n for n, w in ws.items() if (C.adjoint_used(w) if w.is_complex() else pw.transposed_used(w))}

    def step(xi):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            return blk(xi)

    y = step(x)
    assert adjoints() == set()
    y.backward(gy)
    assert adjoints() == {"fc1", "fc2"}
    xi = x.clone().requires_grad_()
    step(xi).backward(gy)
    assert adjoints() == set(ws)
    with torch.no_grad():
        for p in blk.parameters():
            p.mul_(1.25)
    y = step(xi)
    assert C._cache[(id(ws["filter"]), "fp32", True)][1].stamp == C._cache[(id(ws["filter"]), "fp32", False)][1].stamp
    assert all(pw._wcache[(id(w), True)][1] == pw._wcache[(id(w), False)][1] for n, w in ws.items() if n != "filter")
    got = torch.autograd.grad(y, [xi, *ws.values()], gy)
    C.clear_cache()
    pw.clear_cache()
    want = torch.autograd.grad(step(xi), [xi, *ws.values()], gy)
    assert all(torch.equal(torch.view_as_real(a) if a.is_complex() else a, torch.view_as_real(b) if b.is_complex() else b) for a, b in zip(got, want))


def test_validation_with_gradients_enabled_packs_no_adjoint(lib_built):
    """The layers outside a native block likewise: the filter by itself, a single convolution, encoder and decoder pairs."""
    import makani_amd as ma
    from makani_amd import contractions as C
    from makani_amd import pointwise as pw

    fwd, inv = ma.RealSHT(16, 32, grid="legendre-gauss"), ma.InverseRealSHT(16, 32, grid="legendre-gauss")
    conv = ma.SpectralConv(fwd, inv, 8, 8, operator_type="dhconv", gain=2.0).cuda()
    one, a, b = (pw.PointwiseConv2d(8, 8).cuda() for _ in range(3))
    x = torch.randn(2, 8, 16, 32, device="cuda", requires_grad=True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        ys = conv(x)[0], one(x), pw.conv_gelu_conv_trainable(x, a, b)
    used = lambda: [C.adjoint_used(conv.weight), *(pw.transposed_used(m.weight) for m in (one, a, b))]
    assert used() == [False] * 4
    for y in ys:
        y.float().sum().backward()
    assert used() == [True] * 4


def test_batches_past_the_row_limit_are_refused(lib_built):
    """A batch whose rows do not fit the spectral layout's 31-bit row length is refused before anything is launched."""
    import ctypes

    import makani_amd as ma
    from makani_amd import block as nb
    from makani_amd._lib import lib

    sht, isht = ma.RealSHT(16, 32, grid="legendre-gauss"), ma.InverseRealSHT(16, 32, grid="legendre-gauss")
    blk = make_block(sht, isht, 16, 2.0)
    x = torch.randn(1, 16, 16, 32, device="cuda").to(torch.bfloat16)
    with torch.no_grad():
        c = nb._Call(blk, x, nb.block_params(blk))
        huge = 1 << 62
        for batch in ((1 << 25) + 1, 1 << 26, (1 << 31) - 1):        # from 2^29 rows on
            c.b.batch = batch
            assert lib.sfno_block_forward(ctypes.byref(c.b), 0, x.data_ptr(), x.data_ptr(), x.data_ptr(), huge, x.data_ptr(), huge, c.stream) == -1
    torch.cuda.synchronize()


class Rolled(nn.Module):
    """(a factor would not do: the norms take those of the layers in front of them out again)"""

    def forward(self, w):
        return w.roll(1, 0)


@pytest.mark.parametrize("where", ["filter.filter", "norm0", "norm1", "mlp.fwd.0", "mlp.fwd.3", "outer_skip"])
def test_parametrised_members(lib_built, where):
    """A parameter that its module computes is read as the module computes it, in training and in inference, native or not."""
    import makani_amd as ma

    print(f"case parametrised {where}", flush=True)
    torch.manual_seed(8)
    sht, isht = ma.RealSHT(16, 32, grid="legendre-gauss"), ma.InverseRealSHT(16, 32, grid="legendre-gauss")
    blk = make_block(sht, isht, 16, 2.0)
    x = torch.randn(2, 16, 16, 32, device="cuda").to(torch.bfloat16)
    gy = torch.randn_like(x)
    m = blk.get_submodule(where)
    nn.utils.parametrize.register_parametrization(m, "weight", Rolled())
    rolled = passes(blk, x, gy, True)
    ref = passes(blk, x.float(), gy.float(), False)
    assert rel(rolled["y"], ref["y"]) < 1.5e-2
    g = f"{where}.parametrizations.weight.original"
    assert rel(rolled[g], ref[g]) < 1.5e-2
    with torch.inference_mode(), torch.autocast("cuda", dtype=torch.bfloat16):
        assert rel(blk.eval()(x), ref["y"]) < 1.5e-2
    # (the test sees the order)
    nn.utils.parametrize.remove_parametrizations(m, "weight", leave_parametrized=False)
    assert rel(passes(blk.train(), x.float(), gy.float(), False)["y"], ref["y"]) > 3e-2


def test_weight_norm_in_the_mlp(lib_built):
    """weight_norm replaces the parameter by an attribute that a hook sets before each call."""
    import warnings

    import makani_amd as ma

    torch.manual_seed(9)
    sht, isht = ma.RealSHT(16, 32, grid="legendre-gauss"), ma.InverseRealSHT(16, 32, grid="legendre-gauss")
    blk = make_block(sht, isht, 16, 2.0)
    x = torch.randn(2, 16, 16, 32, device="cuda").to(torch.bfloat16)
    gy = torch.randn_like(x)
    with warnings.catch_warnings():
        warnings.simplefilter("ignore")
        nn.utils.weight_norm(blk.mlp.fwd[0])
    with torch.no_grad():
        blk.mlp.fwd[0].weight_g.mul_(3.0)
    got, ref = passes(blk, x, gy, True), passes(blk, x.float(), gy.float(), False)
    assert rel(got["y"], ref["y"]) < 1.5e-2 and rel(got["mlp.fwd.0.weight_g"], ref["mlp.fwd.0.weight_g"]) < 1.5e-2


def test_hooks_on_single_members(lib_built):
    """A hook on any one member is called in training: the block then runs its modules."""
    import makani_amd as ma

    torch.manual_seed(10)
    sht, isht = ma.RealSHT(16, 32, grid="legendre-gauss"), ma.InverseRealSHT(16, 32, grid="legendre-gauss")
    blk = make_block(sht, isht, 16, 2.0)
    x = torch.randn(1, 16, 16, 32, device="cuda").to(torch.bfloat16)
    gy = torch.randn_like(x)
    names = ["filter", "filter.filter", "norm0", "act_layer0", "mlp", "mlp.fwd", *(f"mlp.fwd.{i}" for i in range(len(blk.mlp.fwd))), "norm1", "outer_skip"]
    for name in names:
        for register in ("register_forward_hook", "register_forward_pre_hook"):
            seen = []
            handle = getattr(blk.get_submodule(name), register)(lambda *a: seen.append(1))
            passes(blk, x, gy, True)
            handle.remove()
            assert seen, (name, register)


def test_members_of_wrapped_modules(lib_built):
    """member() and has_member() find what attribute look-up finds: tables, class attributes, instance attributes and what a wrapper hands on."""
    from makani_amd.block import has_member, member

    class Wrapper(nn.Module):
        def __init__(self, inner):
            super().__init__()
            self.inner = inner

        def __getattr__(self, name):
            try:
                return super().__getattr__(name)
            except AttributeError:
                return getattr(super().__getattr__("inner"), name)

    conv = nn.Conv2d(3, 4, 1, bias=False)
    conv.note = "here"
    conv.register_buffer("table", torch.zeros(2))
    for m in (conv, Wrapper(conv)):
        for name in ("weight", "bias", "table", "note", "in_channels", "forward"):
            assert has_member(m, name)
            a, b = member(m, name), getattr(m, name)
            assert a is b or a == b, name
        assert not has_member(m, "absent")
        with pytest.raises(AttributeError):
            member(m, "absent")
    assert member(Wrapper(conv), "inner") is conv
