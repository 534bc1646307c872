"""Spectral losses on the HIP transform: GeometricH1Loss (makani/utils/losses.py:268-360).

The reference transforms `prd - tar` (and `tar`) with RealSHT(*img_shape, grid="equiangular"), reduces the coefficients
to a per-degree power |c_l0|^2 + 2 sum_{m>0} |c_lm|^2 and weights the degrees with 1 (L2 part) and l(l+1) (H1 part).
Here the power comes from one kernel that reads the output of the Legendre analysis in place (no pass to the reference
coefficient layout, no intermediate tensors of the coefficients' size); its gradient feeds the adjoint transform.
"""
import torch
from torch import nn
from torch.autograd.function import once_differentiable

from ._lib import lib, check
from .sht import RealSHT, _ptr, _stream_ptr as _stream


class _DegreePowerFn(torch.autograd.Function):
    """spectral-layout coefficients [mmax, lmax, ld] -> power [rows, lmax]."""

    @staticmethod
    def forward(ctx, spec, rows, lmax, mmax):
        spec = spec.contiguous()
        power = torch.empty((rows, lmax), dtype=torch.float32, device=spec.device)
        check(lib.sfno_degree_power(_ptr(spec), _ptr(power), rows, lmax, mmax, _stream(spec.device)), "sfno_degree_power")
        ctx.save_for_backward(spec)
        ctx.cfg = (rows, lmax, mmax)
        return power

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        (spec,) = ctx.saved_tensors
        rows, lmax, mmax = ctx.cfg
        g = g.float().contiguous()
        gspec = torch.empty_like(spec)
        check(lib.sfno_degree_power_grad(_ptr(spec), _ptr(g), _ptr(gspec), rows, lmax, mmax, _stream(spec.device)), "sfno_degree_power_grad")
        return gspec, None, None, None


class _DegreeNormFn(torch.autograd.Function):
    """spectral-layout coefficients [mmax, lmax, ld] of batch * channels rows -> norms [batch] of GeometricH1Loss."""

    @staticmethod
    def forward(ctx, spec, weights, batch, channels, alpha, squared):
        mmax, lmax, _ = spec.shape
        sums = torch.empty((batch, 2), dtype=torch.float32, device=spec.device)
        norms = torch.empty((batch,), dtype=torch.float32, device=spec.device)
        nbytes = lib.sfno_degree_norm_workspace_bytes(batch, channels, lmax)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=spec.device)
        check(lib.sfno_degree_norm(_ptr(spec), _ptr(weights), _ptr(sums), _ptr(norms), batch, channels, lmax, mmax, alpha, squared, _ptr(ws), nbytes,
                                   _stream(spec.device)), "sfno_degree_norm")
        ctx.save_for_backward(spec, weights, sums)
        ctx.cfg = (batch, channels, lmax, mmax, alpha, squared)
        return norms

    @staticmethod
    @once_differentiable
    def backward(ctx, g):
        spec, weights, sums = ctx.saved_tensors
        batch, channels, lmax, mmax, alpha, squared = ctx.cfg
        g = g.float().contiguous()
        gspec = torch.empty_like(spec)
        check(lib.sfno_degree_norm_grad(_ptr(spec), _ptr(weights), _ptr(sums), _ptr(g), _ptr(gspec), batch, channels, lmax, mmax, alpha, squared,
                                        _stream(spec.device)), "sfno_degree_norm_grad")
        return gspec, None, None, None, None, None


class _PairNormsFn(torch.autograd.Function):
    """Norms [batch] of x - x2 and of x2, differentiable with respect to x: the analyses of both share one Legendre stage."""

    @staticmethod
    def forward(ctx, x, x2, weights, sht, ld, alpha, squared):
        dev, batch = x.device, x.shape[0]
        channels = x.numel() // (batch * sht.nlat * sht.nlon)
        # (two tensors: the backward keeps the first alone)
        spec, spec2 = (torch.empty(sht.spectral_shape(batch * channels), dtype=torch.float32, device=dev) for _ in range(2))
        # the Fourier coefficients, and in their place the powers afterwards
        need = lib.sfno_degree_norm_pair_workspace_bytes(batch, channels, sht.lmax)
        nbytes = max(4 * sht.mmax * sht.nlat * ld, need)
        ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
        sums = torch.empty((2 * batch, 2), dtype=torch.float32, device=dev)
        norms, norms2 = (torch.empty((batch,), dtype=torch.float32, device=dev) for _ in range(2))
        s = _stream(dev)
        check(lib.sfno_sht_analysis_pair(sht.plan(dev).handle, _ptr(x), _ptr(x2), _ptr(spec), _ptr(spec2), batch * channels, _ptr(ws), nbytes, s),
              "sfno_sht_analysis_pair")
        check(lib.sfno_degree_norm_pair(_ptr(spec), _ptr(spec2), _ptr(weights), _ptr(sums), _ptr(norms), _ptr(norms2), batch, channels, sht.lmax, sht.mmax, alpha,
                                        squared, _ptr(ws), nbytes, s), "sfno_degree_norm_pair")
        ctx.save_for_backward(spec, weights, sums)
        ctx.mark_non_differentiable(norms2)
        ctx.sht, ctx.shape, ctx.cfg = sht, x.shape, (batch, channels, alpha, squared)
        return norms, norms2

    @staticmethod
    @once_differentiable
    def backward(ctx, g, _):
        spec, weights, sums = ctx.saved_tensors
        sht, (batch, channels, alpha, squared) = ctx.sht, ctx.cfg
        g = g.float().contiguous()
        gx = torch.empty(ctx.shape, dtype=torch.float32, device=spec.device)
        plan = sht.plan(spec.device, adjoint=True)
        ws, nbytes = sht.workspace(plan, batch * channels, spec.device)
        check(lib.sfno_degree_norm_grad_field(plan.handle, _ptr(spec), _ptr(weights), _ptr(sums), _ptr(g), _ptr(gx), batch, channels, alpha, squared, _ptr(ws), nbytes,
                                              _stream(spec.device)), "sfno_degree_norm_grad_field")
        return gx, None, None, None, None, None, None


def degree_power(sht, x):
    """|c_l0|^2 + 2 sum_{m>0} |c_lm|^2 of sht(x) for every leading index: x [..., nlat, nlon] -> [..., lmax]."""
    lead = x.shape[:-2]
    rows = 1
    for n in lead:
        rows *= int(n)
    if rows == 0:
        return x.new_zeros((*lead, sht.lmax), dtype=torch.float32)
    spec = sht.analysis(x)
    return _DegreePowerFn.apply(spec, rows, sht.lmax, sht.mmax).reshape(*lead, sht.lmax)


class GeometricH1Loss(nn.Module):
    """Weighted H1 loss on the sphere; `alpha` balances the L2 and H1 seminorms (makani/utils/losses.py:268-360)."""

    def __init__(self, img_shape, p=2.0, size_average=False, reduction=True, absolute=False, squared=False, alpha=0.5):
        super().__init__()
        self.reduction = reduction
        self.size_average = size_average
        self.absolute = absolute
        self.squared = squared
        self.alpha = alpha
        self.sht = RealSHT(*img_shape, grid="equiangular").float()
        h1_weights = torch.arange(self.sht.lmax).float()
        self.register_buffer("h1_weights", h1_weights * (h1_weights + 1))

    def _direct(self, x):
        """Whether the kernels form the norms of x directly: a batch of channels of fields, the weights as they were registered."""
        sht, w = self.sht, self.h1_weights
        return type(sht) is RealSHT and x.dim() >= 3 and x.numel() > 0 and x.is_cuda and isinstance(self.alpha, (int, float)) \
            and w.shape == (sht.lmax,) and w.dtype == torch.float32 and w.device == x.device and w.is_contiguous() and not w.requires_grad

    def _norm_pair(self, prd, tar):
        """Norms of prd - tar and of tar: one pass of the transform over both where the target needs no gradient, else one after the other."""
        if type(self)._norms is GeometricH1Loss._norms and isinstance(prd, torch.Tensor) and isinstance(tar, torch.Tensor) and self._direct(prd) \
                and not (tar.requires_grad and torch.is_grad_enabled()) and self.sht.takes_diff(prd, tar):
            sht = self.sht
            ld = int(lib.sfno_sht_analysis_pair_ld(sht.plan(prd.device).handle, prd.numel() // (sht.nlat * sht.nlon)))
            if ld:
                return _PairNormsFn.apply(prd, tar, self.h1_weights, sht, ld, float(self.alpha), bool(self.squared))
        return self._norms(prd, tar), self._norms(tar)

    def _norms(self, x, minus=None):
        """Norms of x, or of x - minus."""
        sht, w = self.sht, self.h1_weights
        if minus is not None and not (isinstance(x, torch.Tensor) and isinstance(minus, torch.Tensor)):
            x, minus = x - minus, None         # a number in place of one of the fields
        if self._direct(x) and (minus is None or minus.shape == x.shape):
            spec = sht.analysis(x) if minus is None else sht.analysis_diff(x, minus)
            rows = x.numel() // (sht.nlat * sht.nlon)
            return _DegreeNormFn.apply(spec, w, x.shape[0], rows // x.shape[0], float(self.alpha), bool(self.squared))
        if minus is not None:
            x = x - minus
        num_examples = x.size()[0]
        norm2 = degree_power(self.sht, x)
        l2_norm2 = norm2.reshape(num_examples, -1).sum(dim=-1)
        h1_norm2 = (norm2 * self.h1_weights).reshape(num_examples, -1).sum(dim=-1)
        if not self.squared:
            return self.alpha * torch.sqrt(l2_norm2) + (1 - self.alpha) * torch.sqrt(h1_norm2)
        return self.alpha * l2_norm2 + (1 - self.alpha) * h1_norm2

    def abs(self, prd, tar):
        all_norms = self._norms(prd, tar)
        if self.reduction:
            return torch.mean(all_norms) if self.size_average else torch.sum(all_norms)
        return all_norms

    def rel(self, prd, tar, mask=None):
        diff, norm = self._norm_pair(prd, tar)
        retval = diff / norm
        if mask is not None:
            retval = retval * mask
        if self.reduction:
            if self.size_average:
                retval = torch.mean(retval) if mask is None else torch.sum(retval) / torch.sum(mask)
            else:
                retval = torch.sum(retval)
        return retval

    def forward(self, prd, tar, mask=None):
        if self.absolute:
            return self.abs(prd, tar)
        return self.rel(prd, tar, mask)
