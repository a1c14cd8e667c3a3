"""The ring-polymer action as a differentiable torch function.

``ring_action(x, ring)`` returns U_M of every chain of a ``Ring`` (instantonmod.f90:17-151)
for the concatenated chain coordinates ``x`` (a float64 tensor, chains in the reference
layout (n, ndim, natom) column-major, one after another).  Its backward pass is the
device adjoint (rp_ring_um), and the backward of that backward is the device
forward-over-reverse Hessian-vector product (rp_ring_hvp), so first and second
derivatives of any scalar built from the actions come from the hand-written kernels.
A tensor on the GPU stays there: the library's stream-ordered entry points
(rp_ring_action_stream, rp_ring_hvp_stream and the per-chain weights and dot products) queue
their kernels on torch's current stream, so nothing waits for the host.  CPU tensors, tensors
on another GPU than the ring's, and potentials that live on the host go through the host entry
points.

The Ring is the function's workspace: every evaluation loads x into its device coordinates
and leaves them there (keep an optimised instanton in a Ring of its own).  The gradient made
by the forward pass is kept for the backward pass, so a first derivative costs one adjoint
evaluation in all.
"""
from __future__ import annotations

import ctypes as C

import numpy as np
import torch

from . import _lib as L
from .instanton import Ring


def _host(t: torch.Tensor) -> np.ndarray:
    return np.ascontiguousarray(t.detach().to("cpu", torch.float64).numpy())


def _flat(chains) -> torch.Tensor:
    return torch.from_numpy(np.concatenate([c.reshape(-1) for c in chains]))


def _on_device(ring: Ring, x: torch.Tensor) -> bool:
    # on the ring's own GPU, and no host potential (which has no spec)
    return x.is_cuda and x.device.index == ring.device and ring.pes.spec is not None


def _f64(t: torch.Tensor) -> torch.Tensor:
    return t.detach().to(torch.float64).contiguous()


def _call(name: str, ring: Ring, like: torch.Tensor, *tensors) -> None:
    """One stream-ordered library call on torch's current stream of the tensors' GPU."""
    if torch.cuda.current_device() != like.device.index:  # a default stream is the current GPU's
        with torch.cuda.device(like.device):
            return _call(name, ring, like, *tensors)
    stream = torch.cuda.current_stream(like.device).cuda_stream
    ptrs = [None if t is None else C.c_void_p(t.data_ptr()) for t in tensors]
    L.check(getattr(L.lib(), name)(ring.h, *ptrs, C.c_void_p(stream)))


def _vector(ring: Ring, t: torch.Tensor, what: str) -> torch.Tensor:
    if t.numel() != int(ring.off[-1]):  # the kernels read the ring's chains, whatever the tensor holds
        raise ValueError(f"ring_action: {what} has {t.numel()} values, the ring's chains {int(ring.off[-1])}")
    return _f64(t)


def _um(ring: Ring, x: torch.Tensor):
    """(U_M per chain, the flat adjoint gradient), float64 on x's device"""
    if _on_device(ring, x):
        xd = _vector(ring, x, "x")
        e = torch.empty(ring.nchain, dtype=torch.float64, device=x.device)
        g = torch.empty_like(xd)
        _call("rp_ring_action_stream", ring, x, xd, e, g)
        return e, g
    ring.set_x(ring.unpack(_host(x)))
    g, e = ring.UMforceenergy()
    return torch.as_tensor(e, device=x.device), _flat(g).to(x.device)


def _hvp(ring: Ring, x: torch.Tensor, v: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    """w_c H_c(x) v of every chain, flat, on x's device (float64)"""
    if _on_device(ring, x):
        hv = torch.empty(v.numel(), dtype=torch.float64, device=x.device)
        _call("rp_ring_hvp_stream", ring, x, _vector(ring, x, "x"), _vector(ring, v, "the vector"), _f64(w), hv)
        return hv
    ring.set_x(ring.unpack(_host(x)))
    hv = _flat(ring.hvp(ring.unpack(_host(v)))).to(x.device)
    return _weighted(ring, x, w, hv)


def _chain_index(ring: Ring, device) -> torch.Tensor:
    """the chain of every element of a flat coordinate vector"""
    sizes = torch.as_tensor(np.diff(ring.off), dtype=torch.int64)
    return torch.repeat_interleave(torch.arange(ring.nchain), sizes).to(device)


def _weighted(ring: Ring, x: torch.Tensor, w: torch.Tensor, g: torch.Tensor) -> torch.Tensor:
    """w_c g over every chain (float64)"""
    if _on_device(ring, x):
        out = torch.empty_like(g)
        _call("rp_ring_weight_stream", ring, x, _f64(w), g, out)
        return out
    return w.to(torch.float64)[_chain_index(ring, x.device)] * g


def _dots(ring: Ring, x: torch.Tensor, a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
    """a . b of every chain (float64)"""
    if _on_device(ring, x):
        out = torch.empty(ring.nchain, dtype=torch.float64, device=x.device)
        _call("rp_ring_dot_stream", ring, x, a, _vector(ring, b, "the vector"), out)
        return out
    out = torch.zeros(ring.nchain, dtype=torch.float64, device=x.device)
    return out.index_add_(0, _chain_index(ring, x.device), a * b.to(torch.float64))


class _Action(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, ring):
        e, g = _um(ring, x)
        ctx.ring = ring
        ctx.g = g
        ctx.save_for_backward(x)
        return e.to(x.dtype)

    @staticmethod
    def backward(ctx, gout):
        (x,) = ctx.saved_tensors
        return _ActionGrad.apply(x, gout, ctx.ring, ctx.g), None


class _ActionGrad(torch.autograd.Function):
    """(x, w) -> sum_c w_c grad U_c(x), laid out like x; g = the flat gradient at x (float64,
    on x's device) when the caller already holds it."""

    @staticmethod
    def forward(ctx, x, w, ring, g=None):
        if g is None:
            _, g = _um(ring, x)
        ctx.ring = ring
        ctx.save_for_backward(x, w)
        ctx.g = g
        return _weighted(ring, x, w, g).to(x.dtype)

    @staticmethod
    def backward(ctx, gg):
        x, w = ctx.saved_tensors
        ring = ctx.ring
        # d/dx: sum_c w_c H_c gg_c (the HVP runs at the x of the forward pass); d/dw_c: grad U_c . gg_c
        dx = _hvp(ring, x, gg, w).to(x.dtype) if ctx.needs_input_grad[0] else None
        dw = _dots(ring, x, ctx.g, gg).to(w.dtype) if ctx.needs_input_grad[1] else None
        return dx, dw, None, None


def ring_action(x: torch.Tensor, ring: Ring) -> torch.Tensor:
    """U_M of every chain of ``ring`` at ``x`` (shape (sum_c n_c * ndof,)), differentiable
    twice: gradients from the adjoint kernel, second derivatives from its HVP."""
    return _Action.apply(x, ring)
