"""Pointwise tail of the SFNO block on the HIP kernels, for bfloat16 NCHW activations.

1x1 convolutions with fused bias / exact GELU / "+ scale * addend + shift" epilogue, and
instance norm split into its statistics (a per-(b, c) scale and shift) and their application.
These replace the nn.Conv2d(kernel_size=1) / nn.InstanceNorm2d / nn.GELU sequences of
makani/models/networks/sfnonet.py:246-262 and makani/models/common/layers.py:86-216 on the
inference path under bf16 autocast.  In training the plain convolution (with its bias) has a backward on the HIP
kernels -- conv1x1_trainable, the forward of PointwiseConv2d when a gradient is asked for --, convolution -> GELU -> convolution
has one (conv_gelu_conv_trainable), and so has a whole block (block.py); the other epilogues have none.
"""
import ctypes
import weakref

import torch

from . import _lib
from ._lib import lib, check
from .sht import _stream_ptr as _stream

ACT = {None: _lib.ACT_NONE, "none": _lib.ACT_NONE, "gelu": _lib.ACT_GELU}

# (id(parameter), transposed) -> (weakref, stamp, packed bf16 [O, Kpad], stream it was packed on, handles of the streams that may use it)
_wcache = {}


def _ptr(t):
    return t.data_ptr() if t is not None else None


def _order(p, packed_on, streams):
    """Puts the current stream, the first time it uses p, behind the stream that packed it, and keeps p's memory until its work is done.
    (A capture is entered with the device idle; work outside it cannot be waited for inside.)"""
    if torch.cuda.is_current_stream_capturing():
        return
    s = torch.cuda.current_stream(p.device)
    s.wait_stream(packed_on)
    p.record_stream(s)
    streams.add(s.cuda_stream)


def packed_weight(weight, transposed=False, both=False):
    """MFMA operand stream of a 1x1 convolution weight ([O, K, 1, 1] or [O, K]), or of its transpose (the weight of the
    convolution's input gradient); cached per parameter and rebuilt when the parameter changes.

    both: the transpose, which the input gradient will ask for, is packed by the same launch."""
    key = (id(weight), transposed)
    # (tensors made under inference_mode carry no version counter: they are packed once per tensor object)
    stamp = (weight.data_ptr(), -1 if weight.is_inference() else weight._version, weight.device)
    hit = _wcache.get(key)
    if hit is not None and hit[0]() is weight and hit[1] == stamp:
        if torch._C._cuda_getCurrentRawStream(weight.device.index) not in hit[4]:
            _order(*hit[2:])
        return hit[2]
    w = weight.detach().reshape(weight.shape[0], -1).float().contiguous()
    O, K = (w.shape[1], w.shape[0]) if transposed else w.shape
    p = torch.empty(lib.sfno_pointwise_weight_elems(O, K), dtype=torch.bfloat16, device=w.device)
    s = torch.cuda.current_stream(w.device)

    def keep(key, p):
        _wcache[key] = (weakref.ref(weight, lambda _, k=key: _wcache.pop(k, None)), stamp, p, s, {s.cuda_stream})

    if both and not transposed:
        pt = torch.empty(lib.sfno_pointwise_weight_elems(K, O), dtype=torch.bfloat16, device=w.device)
        check(lib.sfno_pointwise_pack_weight_both(_ptr(w), _ptr(p), _ptr(pt), O, K, s.cuda_stream), "sfno_pointwise_pack_weight_both")
        keep((id(weight), True), pt)
    else:
        pack = lib.sfno_pointwise_pack_weight_transposed if transposed else lib.sfno_pointwise_pack_weight
        check(pack(_ptr(w), _ptr(p), O, K, s.cuda_stream), "sfno_pointwise_pack_weight")
    keep(key, p)
    return p


def transposed_used(weight):
    """Whether a backward pass has asked for the weight's transpose: then the forwards that record gradients pack it along with the weight."""
    hit = _wcache.get((id(weight), True))
    return hit is not None and hit[0]() is weight


def clear_cache(weight=None):
    """Forgets the packed copy of `weight` (of every weight if None); needed only after writes through ``param.data``, which
    the version stamp of the cache does not see."""
    if weight is None:
        _wcache.clear()
    else:
        _wcache.pop((id(weight), False), None)
        _wcache.pop((id(weight), True), None)


def supported(x):
    """Whether the fused kernels take this activation tensor."""
    return x.is_cuda and x.dim() == 4 and x.dtype == torch.bfloat16 and (x.shape[2] * x.shape[3]) % 8 == 0 and x.shape[2] * x.shape[3] >= 8


def _dense(x):
    """x contiguous and on a 16-byte boundary, as the kernels load it; a view into the middle of a buffer is copied."""
    x = x.contiguous()
    return x if x.data_ptr() % 16 == 0 else x.clone()


def _vector(t):
    """A parameter as the kernels read it: float32 and contiguous (None where there is none)."""
    return t if t is None or (t.dtype == torch.float32 and t.is_contiguous()) else t.detach().float().contiguous()


def conv1x1(x, weight, bias=None, act=None, addend=None, add_scale=None, add_shift=None):
    """act(conv1x1(x, weight) + bias) + add_scale * addend + add_shift  ->  bf16 [B, O, H, W]."""
    return _conv1x1(x, weight, False, bias, act, addend, add_scale, add_shift)


def _conv1x1(x, weight, transposed, bias=None, act=None, addend=None, add_scale=None, add_shift=None, both=False):
    O, K_weight = (weight.shape[1], weight.shape[0]) if transposed else weight.shape[:2]
    if not supported(x):
        raise RuntimeError("the fused pointwise kernels take contiguous bfloat16 NCHW HIP tensors with H*W a multiple of 8")
    x = _dense(x)
    B, K, H, W = x.shape
    if K_weight != K:
        raise RuntimeError(f"conv1x1: input has {K} channels, weight expects {K_weight}")
    pw = packed_weight(weight, transposed, both)
    y = torch.empty((B, O, H, W), dtype=torch.bfloat16, device=x.device)
    bias = _vector(bias)
    if addend is not None:
        if addend.shape != y.shape or addend.dtype != torch.bfloat16:
            raise RuntimeError("conv1x1: addend must be a bfloat16 tensor of the output's shape")
        addend = _dense(addend)
        if add_scale is not None:
            add_scale = add_scale.float().contiguous()
            add_shift = add_shift.float().contiguous()
            assert add_scale.numel() == B * O and add_shift.numel() == B * O
    check(
        lib.sfno_pointwise_conv(_ptr(x), _ptr(pw), _ptr(bias), _ptr(y), B, K, O, H * W, ACT[act], _ptr(addend), _ptr(add_scale),
                                _ptr(add_shift), _stream(x.device)),
        "sfno_pointwise_conv",
    )
    return y


def norm_mlp(x, scale, shift, w1, b1, w2, b2):
    """conv1x1(gelu(conv1x1(gelu(scale[b, c] * x + shift[b, c]), w1) + b1), w2) + b2 -> bf16 [B, E, H, W] in one kernel (inference);
    x has E <= 384 channels, a multiple of 8, and w1 [H, E] a multiple of 16 rows."""
    if not supported(x):
        raise RuntimeError("the fused pointwise kernels take contiguous bfloat16 NCHW HIP tensors with H*W a multiple of 8")
    x = _dense(x)
    B, E, H, W = x.shape
    hidden = w1.shape[0]
    if w1.reshape(hidden, -1).shape[1] != E or tuple(w2.shape[:2]) != (E, hidden) or scale.numel() != B * E or shift.numel() != B * E:
        raise RuntimeError(f"norm_mlp: weights {tuple(w1.shape)} and {tuple(w2.shape)} do not fit {E} channels")
    y = torch.empty_like(x)
    scale, shift, b1, b2 = (t.detach().float().contiguous() if t is not None else None for t in (scale, shift, b1, b2))
    check(lib.sfno_pointwise_mlp(_ptr(x), _ptr(scale), _ptr(shift), _ptr(packed_weight(w1)), _ptr(b1), _ptr(packed_weight(w2)), _ptr(b2), _ptr(y), B, E,
                                 hidden, H * W, _stream(x.device)), "sfno_pointwise_mlp")
    return y


def merged_weight(w, ws, scale, shift, bias, batch):
    """The layer w (scale x1 + shift) + ws x2 + bias of each sample as a convolution for conv1x1_cat: packed weights bf16 [batch, n] and biases
    float32 [batch, O]; w, ws [O, K], scale, shift [batch, K] (both None: 1 and 0), bias [O] or None.  Strided operands are read as their values."""
    O, K = w.shape
    if not w.is_cuda or ws.shape != w.shape or (scale is None) != (shift is None) or any(t is not None and t.device != w.device for t in (ws, scale, shift, bias)) \
            or any(t is not None and t.shape != (batch, K) for t in (scale, shift)) or (bias is not None and bias.shape != (O,)):
        raise RuntimeError(f"merged_weight: operands do not fit a weight {tuple(w.shape)} on {w.device} and {batch} samples")
    packed = torch.empty((batch, lib.sfno_pointwise_weight_elems(O, 2 * K)), dtype=torch.bfloat16, device=w.device)
    shifted = torch.empty((batch, O), dtype=torch.float32, device=w.device)
    w, ws, scale, shift, bias = (_vector(t) for t in (w, ws, scale, shift, bias))
    check(lib.sfno_pointwise_merge_weight(_ptr(w), _ptr(ws), _ptr(scale), _ptr(shift), _ptr(bias), _ptr(packed), _ptr(shifted), O, K, batch, _stream(w.device)),
          "sfno_pointwise_merge_weight")
    return packed, shifted


def conv1x1_cat(x1, x2, weight, bias=None, act=None, out=None, packed=None):
    """act(conv1x1(cat([x1, x2], dim=1), weight) + bias) without building the concatenation  ->  bf16 [B, O, H, W];
    weight [O, K1 + K2] (or [O, K1 + K2, 1, 1]); out: a contiguous bf16 tensor of the result's shape to write into; packed: the weight's stream
    where the caller has it (weight is then its shape)."""
    if not (supported(x1) and supported(x2)) or x1.shape[0] != x2.shape[0] or x1.shape[2:] != x2.shape[2:]:
        raise RuntimeError("conv1x1_cat takes two contiguous bfloat16 NCHW HIP tensors of one batch and grid size, H*W a multiple of 8")
    x1, x2 = _dense(x1), _dense(x2)
    B, K1, H, W = x1.shape
    K2 = x2.shape[1]
    O, K = (weight.shape[0], weight.shape[1:].numel()) if packed is None else weight
    if K != K1 + K2:
        raise RuntimeError(f"conv1x1_cat: inputs have {K1} + {K2} channels, weight expects {K}")
    if packed is None:
        pw = packed_weight(weight)
    elif packed.dtype != torch.bfloat16 or not packed.is_contiguous() or packed.device != x1.device or packed.numel() != lib.sfno_pointwise_weight_elems(O, K):
        raise RuntimeError(f"conv1x1_cat: packed is not the stream of a weight [{O}, {K}]")
    else:
        pw = packed
    if out is None:
        y = torch.empty((B, O, H, W), dtype=torch.bfloat16, device=x1.device)
    else:
        if tuple(out.shape) != (B, O, H, W) or out.dtype != torch.bfloat16 or not out.is_contiguous() or out.device != x1.device:
            raise RuntimeError("conv1x1_cat: out must be a contiguous bfloat16 tensor of the result's shape")
        y = out
    bias = _vector(bias)
    check(lib.sfno_pointwise_conv_cat(_ptr(x1), K1, _ptr(x2), K2, _ptr(pw), _ptr(bias), _ptr(y), B, O, H * W, ACT[act], _stream(x1.device)),
          "sfno_pointwise_conv_cat")
    return y


def instance_norm_coeffs(x, gamma=None, beta=None, eps=1e-5):
    """(scale, shift) float32 [B, C] such that instance_norm(x) = scale * x + shift."""
    if not supported(x):
        raise RuntimeError("the fused pointwise kernels take contiguous bfloat16 NCHW HIP tensors with H*W a multiple of 8")
    x = _dense(x)
    B, C, H, W = x.shape
    rows, P = B * C, H * W
    scale = torch.empty((B, C), dtype=torch.float32, device=x.device)
    shift = torch.empty_like(scale)
    nbytes = lib.sfno_instance_norm_workspace_bytes(rows, P)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    g = gamma.detach().float().contiguous() if gamma is not None else None
    b = beta.detach().float().contiguous() if beta is not None else None
    check(
        lib.sfno_instance_norm_coeffs(_ptr(x), _ptr(g), _ptr(b), _ptr(scale), _ptr(shift), rows, C, P, float(eps), _ptr(ws), nbytes, _stream(x.device)),
        "sfno_instance_norm_coeffs",
    )
    return scale, shift


# grids of at most this many pixels are normalised by the moments of the stored field (NORM_SMALL_PIXELS in csrc/sfno_internal.h)
NORM_SMALL_PIXELS = 4096


def instance_norm_coeffs_lat(lat_stats, batch, gamma=None, beta=None, eps=1e-5):
    """(scale, shift) float32 [B, C] from the per-latitude moments [B*C, nlat, 2] that InverseRealSHT.synthesis_with_lat_stats returns."""
    rows, nlat, _ = lat_stats.shape
    C = rows // batch
    scale = torch.empty((batch, C), dtype=torch.float32, device=lat_stats.device)
    shift = torch.empty_like(scale)
    g = gamma.detach().float().contiguous() if gamma is not None else None
    b = beta.detach().float().contiguous() if beta is not None else None
    check(lib.sfno_instance_norm_coeffs_lat(_ptr(lat_stats), _ptr(g), _ptr(b), _ptr(scale), _ptr(shift), rows, C, nlat, float(eps),
                                            _stream(lat_stats.device)), "sfno_instance_norm_coeffs_lat")
    return scale, shift


def scale_shift_act(x, scale, shift, act=None):
    """act(scale[b, c] * x + shift[b, c]) -> bf16, same shape."""
    if not supported(x):
        raise RuntimeError("the fused pointwise kernels take contiguous bfloat16 NCHW HIP tensors with H*W a multiple of 8")
    x = _dense(x)
    B, C, H, W = x.shape
    y = torch.empty_like(x)
    check(lib.sfno_scale_shift_act(_ptr(x), _ptr(scale), _ptr(shift), _ptr(y), B * C, H * W, ACT[act], _stream(x.device)), "sfno_scale_shift_act")
    return y


def conv1x1_weight_grad(gy, x, with_bias):
    """(gweight float32 [O, K], gbias float32 [O] or None) of y = conv1x1(x, weight) + bias for the output gradient gy:
    gweight[o, k] = sum_{b,p} gy[b, o, p] x[b, k, p], gbias[o] = sum_{b,p} gy[b, o, p]; bf16 operands, fp32 sums in a fixed order."""
    if not (supported(x) and supported(gy)) or gy.shape[0] != x.shape[0] or gy.shape[2:] != x.shape[2:]:
        raise RuntimeError("conv1x1_weight_grad takes two contiguous bfloat16 NCHW HIP tensors of one batch and grid size, H*W a multiple of 8")
    x, gy = _dense(x), _dense(gy)
    B, K, H, W = x.shape
    O = gy.shape[1]
    gw = torch.empty((O, K), dtype=torch.float32, device=x.device)
    gb = torch.empty((O,), dtype=torch.float32, device=x.device) if with_bias else None
    nbytes = lib.sfno_pointwise_weight_grad_workspace_bytes(B, K, O, H * W, 1 if with_bias else 0)
    ws = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    check(lib.sfno_pointwise_weight_grad(_ptr(gy), _ptr(x), _ptr(gw), _ptr(gb), B, K, O, H * W, _ptr(ws), nbytes, _stream(x.device)),
          "sfno_pointwise_weight_grad")
    return gw, gb


class _Conv1x1(torch.autograd.Function):
    """y = conv1x1(x, weight) + bias on the HIP kernels, with the three gradients autograd derives for nn.Conv2d(kernel_size=1)
    (makani/models/common/layers.py:95-116,160-216): the input gradient is the same convolution with the transposed weight."""

    @staticmethod
    def forward(ctx, x, weight, bias):
        xb = _dense(x.detach().to(torch.bfloat16))
        ctx.save_for_backward(xb, weight)
        ctx.has_bias = bias is not None
        ctx.x_dtype = x.dtype
        ctx.b_dtype = bias.dtype if bias is not None else None
        # (the parameter itself goes in: its packed copy is cached per parameter object and version)
        return _conv1x1(xb, weight, False, bias, both=ctx.needs_input_grad[0] and transposed_used(weight))

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, gy):
        xb, weight = ctx.saved_tensors
        gy = _dense(gy.to(torch.bfloat16))
        gx = gw = gb = None
        if ctx.needs_input_grad[0]:
            gx = _conv1x1(gy, weight, True).to(ctx.x_dtype)
        if ctx.needs_input_grad[1] or (ctx.has_bias and ctx.needs_input_grad[2]):
            gw, gb = conv1x1_weight_grad(gy, xb, ctx.has_bias)
            gw = gw.reshape(weight.shape).to(weight.dtype)
            if gb is not None:
                gb = gb.to(ctx.b_dtype)
        return gx, gw, gb


class _ConvGeluConv(torch.autograd.Function):
    """y = W2 gelu(W1 x + b1) + b2 (makani/models/common/layers.py:95-116: the encoder's and the decoder's two convolutions): the first
    convolution stores its output before and after the GELU, the input gradient of the second one is multiplied by the GELU's derivative
    where it is stored."""

    @staticmethod
    def forward(ctx, x, w1, b1, w2, b2):
        xb = _dense(x.detach().to(torch.bfloat16))
        B, K, H, W = xb.shape
        O = w1.shape[0]
        if w1.shape[1] != K or w2.shape[1] != O:
            raise RuntimeError(f"conv1x1: input has {K} channels, weights expect {w1.shape[1]} and {w2.shape[1]} (of {O})")
        z = torch.empty((B, O, H, W), dtype=torch.bfloat16, device=x.device)
        a = torch.empty_like(z)
        bias = _vector(b1)
        need = ctx.needs_input_grad
        check(lib.sfno_pointwise_conv_gelu(_ptr(xb), _ptr(packed_weight(w1, both=need[0] and transposed_used(w1))), _ptr(bias), _ptr(a), _ptr(z), B, K, O, H * W,
                                           _stream(x.device)), "sfno_pointwise_conv_gelu")
        ctx.save_for_backward(xb, z, a, w1, w2)
        ctx.biases = (b1 is not None, b2 is not None)
        ctx.x_dtype = x.dtype
        return _conv1x1(a, w2, False, b2, both=any(need[:3]) and transposed_used(w2))

    @staticmethod
    @torch.autograd.function.once_differentiable
    def backward(ctx, gy):
        xb, z, a, w1, w2 = ctx.saved_tensors
        gy = _dense(gy.to(torch.bfloat16))
        need = ctx.needs_input_grad
        gx = gw1 = gb1 = gw2 = gb2 = None
        if need[3] or need[4]:
            gw2, gb2 = conv1x1_weight_grad(gy, a, ctx.biases[1])
            gw2 = gw2.reshape(w2.shape)
        if need[0] or need[1] or need[2]:
            B, O, H, W = gy.shape
            gz = torch.empty_like(z)
            check(lib.sfno_pointwise_conv_gelu_grad(_ptr(gy), _ptr(packed_weight(w2, transposed=True)), _ptr(z), _ptr(gz), B, O, z.shape[1], H * W,
                                                    _stream(gy.device)), "sfno_pointwise_conv_gelu_grad")
            if need[1] or need[2]:
                gw1, gb1 = conv1x1_weight_grad(gz, xb, ctx.biases[0])
                gw1 = gw1.reshape(w1.shape)
            if need[0]:
                gx = _conv1x1(gz, w1, True).to(ctx.x_dtype)
        return gx, gw1, gb1, gw2, gb2


def conv_gelu_conv_trainable(x, conv1, conv2):
    """conv2(gelu(conv1(x))) -> bf16, differentiable; None where the kernels do not serve the parameters (float32 on the device)."""
    params = [p for p in (conv1.weight, conv1.bias, conv2.weight, conv2.bias) if p is not None]
    if not all(p.dtype == torch.float32 and p.is_cuda for p in params):
        return None
    return _ConvGeluConv.apply(x, conv1.weight, conv1.bias, conv2.weight, conv2.bias)


def trainable_active(x):
    """Whether PointwiseConv2d routes this call through the HIP kernels: a gradient is being recorded and the activations are
    bf16 (or will be under bf16 autocast) HIP tensors the kernels take."""
    if not torch.is_grad_enabled() or not x.is_cuda or x.dim() != 4:
        return False
    bf16 = x.dtype == torch.bfloat16 or (torch.is_autocast_enabled() and torch.get_autocast_dtype("cuda") == torch.bfloat16)
    return bf16 and (x.shape[2] * x.shape[3]) % 8 == 0 and x.shape[2] * x.shape[3] >= 8


def conv1x1_trainable(x, weight, bias=None):
    """conv1x1(x, weight) + bias -> bf16, differentiable with respect to x, weight and bias (HIP kernels in both directions)."""
    return _Conv1x1.apply(x, weight, bias)


class PointwiseConv2d(torch.nn.Conv2d):
    """nn.Conv2d(kernel_size=1) whose training forward and backward under bf16 run on the HIP kernels; every other call (fp32,
    CPU, no gradient) is nn.Conv2d.  Same parameters and state-dict keys."""

    def __init__(self, in_channels, out_channels, bias=True):
        super().__init__(in_channels, out_channels, 1, bias=bias)

    def forward(self, x):
        if trainable_active(x) and (x.requires_grad or self.weight.requires_grad):
            return conv1x1_trainable(x, self.weight, self.bias)
        return super().forward(x)
