"""Differentiable transforms for PyTorch over the library's device entry points.

``fftn(x, rank, weight=None, inverse=False)`` returns ``weight * F(x)`` where
F is the forward DFT over the last ``rank`` dims (or the unnormalised
backward DFT with ``inverse=True``) and ``weight`` is an optional real FP32
tensor of the transform's shape, broadcast over the batch.

Backward is the hand-written adjoint: for y = W . F x the gradient is
F^H (W . g), the unnormalised opposite-direction transform with W fused into
its first pass's loads (fftamd_c2c_weighted_dev), so the backward costs one
transform and no extra elementwise pass.  PyTorch's convention for complex
inputs is followed (grad = 2 dL/d conj(x) for a real loss).  A gradient for
``weight`` (Re sum_batch conj(g) . F x) is produced when it requires grad.
"""
from __future__ import annotations

import ctypes
import math

import torch

from ._lib import last_error, load, stream_handle


def _check(x, rank):
    if not x.is_cuda or x.dtype != torch.complex64:
        raise TypeError("complex64 CUDA/HIP tensor expected")
    if rank < 1 or rank > 3 or x.dim() < rank:
        raise ValueError("bad rank")


def weighted_transform(x, rank, inverse=False, w_in=None, w_out=None, out=None):
    """out = w_out . F(w_in . x) on the current stream (no autograd)."""
    _check(x, rank)
    x = x.contiguous()
    dims = x.shape[x.dim() - rank:]
    batch = x.numel() // max(1, math.prod(dims))
    if out is None:
        out = torch.empty_like(x)
    for w in (w_in, w_out):
        if w is not None and (w.dtype != torch.float32 or not w.is_cuda or w.shape != dims
                              or not w.is_contiguous()):
            raise ValueError("weights must be contiguous float32 CUDA/HIP tensors of the transform shape")
    if batch == 0:
        return out
    cd = (ctypes.c_uint * rank)(*dims)
    rc = load().fftamd_c2c_weighted_dev(
        rank, cd, batch, x.data_ptr(), out.data_ptr(), 1 if inverse else 0,
        w_in.data_ptr() if w_in is not None else None, w_out.data_ptr() if w_out is not None else None,
        stream_handle(x.device))
    if rc != 0:
        raise RuntimeError(f"fftamd weighted transform failed: {last_error()}")
    return out


def weight_gradient(g, fx, rank):
    """Re sum over the batch of conj(g) . fx, one float per point of a transform (no autograd)."""
    _check(fx, rank)
    dims = fx.shape[fx.dim() - rank:]
    # a lazily conjugated or negated gradient is made plain: the kernel reads its memory
    g, fx = g.resolve_conj().resolve_neg().contiguous(), fx.contiguous()
    if g.dtype != fx.dtype or g.shape != fx.shape or g.device != fx.device:
        raise ValueError("g must match fx")
    points = math.prod(dims)
    if fx.numel() == 0:
        return torch.zeros(dims, dtype=torch.float32, device=fx.device)
    gw = torch.empty(dims, dtype=torch.float32, device=fx.device)
    cd = (ctypes.c_uint * rank)(*dims)
    rc = load().fftamd_weight_grad_dev(rank, cd, fx.numel() // points, g.data_ptr(), fx.data_ptr(), gw.data_ptr(),
                                       stream_handle(fx.device))
    if rc != 0:
        raise RuntimeError(f"fftamd weight gradient failed: {last_error()}")
    return gw


class _WeightedFFT(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, weight, rank, inverse):
        y = weighted_transform(x, rank, inverse=inverse, w_out=weight)
        ctx.rank = rank
        ctx.inverse = inverse
        ctx.has_w = weight is not None
        if weight is None:
            ctx.save_for_backward()
        elif weight.requires_grad:
            ctx.save_for_backward(weight, x)
        else:
            ctx.save_for_backward(weight)
        return y

    @staticmethod
    def backward(ctx, g):
        saved = ctx.saved_tensors
        w = saved[0] if ctx.has_w else None
        x = saved[1] if len(saved) > 1 else None
        g = g.contiguous()
        gx = None
        if ctx.needs_input_grad[0]:
            # adjoint of W . F is F^H . W: opposite direction, weights on the load
            gx = weighted_transform(g, ctx.rank, inverse=not ctx.inverse, w_in=w)
        gw = None
        if ctx.has_w and ctx.needs_input_grad[1]:
            fx = weighted_transform(x, ctx.rank, inverse=ctx.inverse)
            if torch.is_grad_enabled():  # create_graph: torch records the product
                prod = (torch.conj(g) * fx).real
                gw = prod.reshape(-1, *w.shape).sum(0)
            else:
                gw = weight_gradient(g, fx, ctx.rank)
        return gx, gw, None, None


def fftn(x, rank: int = 3, weight=None, inverse: bool = False):
    """Differentiable weight . F(x) over the last `rank` dims (see module doc)."""
    return _WeightedFFT.apply(x, weight, rank, inverse)


def fft3(x, weight=None):
    return fftn(x, 3, weight, False)


def ifft3_unnormalised(x, weight=None):
    return fftn(x, 3, weight, True)
