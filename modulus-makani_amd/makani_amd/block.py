"""One SFNO block per native call: filter -> norm0 -> GELU -> MLP -> norm1 -> + outer skip (makani/models/networks/sfnonet.py:239-267)
with every kernel enqueued by sfno_block_forward / sfno_block_backward, for bfloat16 activations.

Inference runs it on buffers that the call needs anyway; training keeps the tensors the backward reads in one buffer.  The
parameters stay those of the PyTorch modules; packed copies come from the caches of contractions.py and pointwise.py.
"""
import ctypes

import torch
import torch.nn as nn
from torch.autograd.function import once_differentiable

from . import _lib
from ._lib import lib, check
from . import pointwise as pw
from .contractions import adjoint_used, packed_for
from .sht import _stream_ptr
from .spectral_convolution import SpectralConv


def _ptr(t):
    return t.data_ptr() if t is not None else None


# The checks of a call read some forty attributes of modules, and for small grids they take longer than the kernels.  nn.Module finds a parameter
# or submodule only after the ordinary look-up has failed (and builds a message where there is none), so these look in its tables first.

def member(m, name):
    """m.name of a module"""
    mods = m._modules
    if name in mods:
        return mods[name]
    params = m._parameters
    return params[name] if name in params else getattr(m, name)


def has_member(m, name):
    """hasattr(m, name) of a module"""
    if type(m).__getattr__ is not nn.Module.__getattr__:
        return hasattr(m, name)
    return name in m._modules or name in m._parameters or name in m._buffers or name in m.__dict__ or hasattr(type(m), name)


def _no_hooks(*mods):
    if torch.nn.modules.module._has_any_global_hook():
        return False
    for m in mods:
        if m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks:
            return False
    return True


def plain_conv(m):
    """A convolution whose forward is known: subclasses (quantisation, adapters) bring their own."""
    return type(m) in (nn.Conv2d, pw.PointwiseConv2d)


def trainable(x, params, *convs):
    """Whether a call with gradients enabled may run on the HIP kernels: something asks for a gradient, and every convolution is one that
    would train on them by itself (nn.Conv2d put in by a user is differentiable twice, the kernels once)."""
    return pw.trainable_active(x) and all(type(m) is pw.PointwiseConv2d for m in convs) and (x.requires_grad or any(p is not None and p.requires_grad for p in params))


def mlp_convs(blk):
    """(fc1, fc2) of a conv -> GELU -> conv MLP, or None."""
    m = [f for f in member(member(blk, "mlp"), "fwd") if not isinstance(f, nn.Identity)]
    ok = len(m) == 3 and plain_conv(m[0]) and plain_conv(m[2]) and type(m[1]) is nn.GELU and m[1].approximate == "none"
    return (m[0], m[2]) if ok else None


def shapes_fit(params, c_in, embed, lmax):
    """Whether the parameters (in the order of block_params) belong to one block: the native calls address all of them by c_in, embed,
    hidden and lmax, so anything else is left to the modules, which raise their own errors."""
    hidden, e = params[2].shape[0], (embed,)
    for p, w in zip(params, ((c_in, embed, lmax), (embed, c_in, 1, 1), (hidden, embed, 1, 1), (hidden,), (embed, hidden, 1, 1), e, e, e, e, e)):
        if p is not None and p.shape != w:
            return False
    return True


def supported(blk, x, filter_weight=None, skip_weight=None, training=False):
    """The block's parameters (true) where the native block serves this block (whose fusable() the caller has checked) and input, else False;
    filter_weight, skip_weight: as of forward(); training: with its gradients, see trainable()."""
    layer, norm0, norm1, act, mlp, skip = (member(blk, n) for n in ("filter", "norm0", "norm1", "act_layer0", "mlp", "outer_skip"))
    conv = member(layer, "filter")
    fwd, inv = member(conv, "forward_transform"), member(conv, "inverse_transform")
    convs = mlp_convs(blk)
    if x.dtype != torch.bfloat16 or x.dim() != 4 or x.shape[0] == 0 or not conv._fused or has_member(conv, "bias") or convs is None:
        return False
    if type(norm0) is not nn.InstanceNorm2d or type(norm1) is not nn.InstanceNorm2d or inv.mmax > inv.nlon // 2 + 1:
        return False
    if type(act) is not nn.GELU or type(conv) is not SpectralConv or not plain_conv(skip):
        return False
    params = _with(block_params(blk, convs), filter_weight, skip_weight)
    if training and not trainable(x, params, *convs, skip):
        return False
    if tuple(x.shape[2:]) != (fwd.nlat, fwd.nlon) or (inv.nlat * inv.nlon) % 8 != 0:
        return False
    if not lib.sfno_sht_io_dtype_supported(fwd.plan(x.device).handle, _lib.DTYPE_BF16) or not lib.sfno_sht_io_dtype_supported(inv.plan(x.device).handle, _lib.DTYPE_BF16):
        return False
    if x.is_contiguous() and x.data_ptr() % 16 != 0:      # a view into the middle of a buffer: the kernels load 16 bytes at a time
        return False
    if not shapes_fit(params, x.shape[1], conv.out_channels, inv.lmax):
        return False
    wf, *rest = [p for p in params if p is not None]
    if wf.dtype != torch.complex64 or not wf.is_cuda:
        return False
    for p in rest:
        if p.dtype != torch.float32 or not p.is_cuda:
            return False
    chain = member(mlp, "fwd")
    return params if _no_hooks(layer, conv, norm0, norm1, act, mlp, chain, *chain, skip) else False


def block_params(blk, convs=None):
    """The block's parameters in the order of _Call: filter, skip, W1, b1, W2, b2, gamma0, beta0, gamma1, beta1 (None where there is none)."""
    fc1, fc2 = convs or mlp_convs(blk)
    n0, n1 = member(blk, "norm0"), member(blk, "norm1")
    return [member(member(member(blk, "filter"), "filter"), "weight"), member(member(blk, "outer_skip"), "weight"),
            *(member(m, n) for m in (fc1, fc2, n0, n1) for n in ("weight", "bias"))]


def _with(params, filter_weight, skip_weight):
    """params with other filter and skip weights in place of the block's own, where there are any."""
    return [params[0] if filter_weight is None else filter_weight, params[1] if skip_weight is None else skip_weight, *params[2:]]


class _Call:
    """The sfno_block structure of one call, and what has to stay alive while it is used.  The values come from `params` alone: the
    modules may hold others by the time of the backward (functional calls, parametrisations).

    training: a forward that records gradients; backward: of the input and the parameters (input_grad) or of the parameters alone."""

    def __init__(self, blk, x, params, backward=False, training=False, input_grad=True):
        conv = member(member(blk, "filter"), "filter")
        fwd, inv = member(conv, "forward_transform"), member(conv, "inverse_transform")
        wf, wskip, w1, b1, w2, b2, g0, be0, g1, be1 = params
        dev = x.device
        b = _lib.Block()
        keep = self.keep = [fwd.plan(dev), inv.plan(dev), packed_for(wf, conv.compute, both=training and adjoint_used(wf, conv.compute)),
                            *(pw.packed_weight(w, both=training and pw.transposed_used(w)) for w in (w1, w2, wskip))]
        b.fwd, b.inv, b.weights = keep[0].handle, keep[1].handle, keep[2].handle
        b.w1, b.w2, b.wskip = (t.data_ptr() for t in keep[3:6])
        if backward:
            adj = [fwd.plan(dev, adjoint=True), inv.plan(dev, adjoint=True), pw.packed_weight(w1, transposed=True), pw.packed_weight(w2, transposed=True)]
            b.fwd_adj, b.inv_adj, b.w1t, b.w2t = adj[0].handle, adj[1].handle, adj[2].data_ptr(), adj[3].data_ptr()
            if input_grad:
                adj += [packed_for(wf, conv.compute, adjoint=True), pw.packed_weight(wskip, transposed=True)]
                b.weights_adj, b.wskipt = adj[4].handle, adj[5].data_ptr()
            keep += adj
        vectors = [t if t is None or t.is_contiguous() else t.detach().contiguous() for t in (b1, b2, g0, be0, g1, be1)]
        keep += vectors
        b.b1, b.b2, b.gamma0, b.beta0, b.gamma1, b.beta1 = (_ptr(t) for t in vectors)
        b.eps0, b.eps1 = member(blk, "norm0").eps, member(blk, "norm1").eps
        b.batch, b.c_in, b.embed, b.hidden = x.shape[0], x.shape[1], conv.out_channels, w1.shape[0]
        self.b = b
        self.P = (inv.nlat, inv.nlon)
        self.stream = _stream_ptr(dev)
        self.offsets = (ctypes.c_int64 * _lib.BLOCK_TENSORS)()

    def forward(self, x, training, out):
        ref = ctypes.byref(self.b)
        nkept, nws = lib.sfno_block_layout(ref, training, self.offsets), lib.sfno_block_workspace_bytes(ref, 0)
        if training or out is None:
            kept = torch.empty(nkept, dtype=torch.uint8, device=x.device)
            at = (ws := torch.empty(nws, dtype=torch.uint8, device=x.device)).data_ptr()
        else:                 # nothing outlives the call: one buffer (pieces of whole 256 bytes)
            kept = torch.empty(nkept + nws, dtype=torch.uint8, device=x.device)
            at = kept.data_ptr() + nkept
        check(lib.sfno_block_forward(ref, training, x.data_ptr(), _ptr(out), kept.data_ptr(), nkept, at, nws, self.stream), "sfno_block_forward")
        return kept


def forward(blk, x, filter_weight=None, skip_weight=None, defer_skip=False, params=None):
    """The block without autograd.  filter_weight, skip_weight: in place of the block's own (params: what supported() returned for them).
    defer_skip: returns (y2, residual, scale, shift) of the last sum scale * y2 + shift + skip(residual) instead of running it."""
    x = x.contiguous()
    c = _Call(blk, x, params or _with(block_params(blk), filter_weight, skip_weight))
    B, E = x.shape[0], c.b.embed
    if not defer_skip:
        out = torch.empty((B, E, *c.P), dtype=torch.bfloat16, device=x.device)
        c.forward(x, 0, out)
        return out
    kept = c.forward(x, 0, None)

    def view(i, shape, dtype):
        n = dtype.itemsize
        for d in shape:
            n *= d
        return kept[c.offsets[i]:c.offsets[i] + n].view(dtype).view(shape)

    coef = view(_lib.BLOCK_COEF1, (2, B, E), torch.float32)
    res = x if c.offsets[_lib.BLOCK_RES] < 0 else view(_lib.BLOCK_RES, (B, x.shape[1], *c.P), torch.bfloat16)
    return view(_lib.BLOCK_Y2, (B, E, *c.P), torch.bfloat16), res, coef[0], coef[1]


class _BlockFn(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, blk, *params):
        x = x.detach().contiguous()
        c = _Call(blk, x, params, training=any(ctx.needs_input_grad))
        out = torch.empty((x.shape[0], c.b.embed, *c.P), dtype=torch.bfloat16, device=x.device)
        kept = c.forward(x, 1, out)
        ctx.blk = blk
        ctx.save_for_backward(x, kept, *params)
        return out

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        x, kept, *params = ctx.saved_tensors
        g = pw._dense(g.to(torch.bfloat16))
        blk, need = ctx.blk, ctx.needs_input_grad
        c = _Call(blk, x, params, backward=True, input_grad=need[0])
        want = [p is not None and n for p, n in zip(params, need[2:])]
        want[2], want[4] = want[2] or want[3], want[4] or want[5]          # a bias gradient comes with its matrix's
        grads = [torch.empty(p.shape, dtype=p.dtype, device=p.device) if w else None for p, w in zip(params, want)]
        gx = torch.empty_like(x) if need[0] else None
        s = _lib.BlockGrads()
        s.gx, s.gfilter = _ptr(gx), _ptr(grads[0])
        s.gwskip, s.gw1, s.gb1, s.gw2, s.gb2, s.ggamma0, s.gbeta0, s.ggamma1, s.gbeta1 = (_ptr(t) for t in grads[1:])
        ref = ctypes.byref(c.b)
        nws = lib.sfno_block_workspace_bytes(ref, 1)
        ws = torch.empty(nws, dtype=torch.uint8, device=x.device)
        check(lib.sfno_block_backward(ref, g.data_ptr(), x.data_ptr(), kept.data_ptr(), kept.numel(), ctypes.byref(s), ws.data_ptr(), nws, c.stream), "sfno_block_backward")
        return (gx, None, *(t if n else None for t, n in zip(grads, need[2:])))


def train(blk, x, params=None):
    """The block with autograd (supported(training=True) holds; params: what it returned)."""
    return _BlockFn.apply(x, blk, *(params or block_params(blk)))
