"""Differentiable wrappers over the C ABI (optional torch.autograd binding).

Every operator of the path is linear, so each backward is the operator's
adjoint, computed by the library's adjoint entry points:
  forward FFT          -> zm_forward_adjoint  (the inverse chain, scale 1)
  inverse FFT (s)      -> zm_inverse_adjoint  (s x the forward chain)
  Laplacian            -> itself (symmetric periodic stencil)
  dx4 / dy4 / dz4      -> zm_dx4_adjoint / zm_dy4_adjoint / zm_dz4_adjoint (the
                          transposed stencil, -dx4)
  spectral multiplier  -> zm_spectral_multiply_adjoint (conjugate multiplier;
                          the real kinds are self-adjoint)
  spectral solve       -> zm_spectral_solve_adjoint (the conjugate multiplier
                          between the same two transforms)
  heat step            -> itself (real multiplier, symmetric Laplacian)
  Poisson misfit       -> the adjoint solve of twice the saved residual; the only
                          operator that saves a tensor for backward
For complex tensors torch passes dL/d(conj y) and expects A^H of it back, which
is exactly the adjoint.
"""
from __future__ import annotations

import torch


def _raw(t):
    """t with its storage in the order and with the values that the library reads:
    contiguous, lazy conjugations and negations carried out."""
    if t.is_conj() or t.is_neg():
        t = t.resolve_conj().resolve_neg()
    return t.contiguous()


class _Forward(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, plan):
        ctx.plan = plan
        return plan.forward(_raw(x))

    @staticmethod
    def backward(ctx, g):
        return ctx.plan.forward_adjoint(_raw(g)), None


class _Inverse(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, plan, scale):
        ctx.plan, ctx.scale = plan, scale
        return plan.inverse(_raw(x), scale)

    @staticmethod
    def backward(ctx, g):
        return ctx.plan.inverse_adjoint(_raw(g), ctx.scale), None, None


class _Laplace(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, plan, scale):
        ctx.plan, ctx.scale = plan, scale
        return plan.laplace(_raw(x), scale)

    @staticmethod
    def backward(ctx, g):
        return ctx.plan.laplace(_raw(g), ctx.scale), None, None


class _Dx4(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, plan, delta):
        ctx.plan, ctx.delta = plan, delta
        return plan.dx4(_raw(x), delta)

    @staticmethod
    def backward(ctx, g):
        return ctx.plan.dx4(_raw(g), ctx.delta, adjoint=True), None, None


class _Dy4(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, plan, delta):
        ctx.plan, ctx.delta = plan, delta
        return plan.dy4(_raw(x), delta)

    @staticmethod
    def backward(ctx, g):
        return ctx.plan.dy4(_raw(g), ctx.delta, adjoint=True), None, None


class _Dz4(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, plan, delta):
        ctx.plan, ctx.delta = plan, delta
        return plan.dz4(_raw(x), delta)

    @staticmethod
    def backward(ctx, g):
        return ctx.plan.dz4(_raw(g), ctx.delta, adjoint=True), None, None


class _Spectral(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, plan, kind, p0, p1, length):
        ctx.args = (plan, kind, p0, p1, length)
        return plan.spectral_multiply(_raw(x), kind, p0, p1, length)

    @staticmethod
    def backward(ctx, g):
        plan, kind, p0, p1, length = ctx.args
        return (plan.spectral_multiply(_raw(g), kind, p0, p1, length, adjoint=True),
                None, None, None, None, None)


class _SpectralSolve(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, plan, *args):
        ctx.plan, ctx.args = plan, args
        return plan.spectral_solve(_raw(x), *args)

    @staticmethod
    def backward(ctx, g):
        return (ctx.plan.spectral_solve(_raw(g), *ctx.args, adjoint=True),) + (None,) * (1 + len(ctx.args))


class _HeatStep(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, plan, *args):
        ctx.plan, ctx.args = plan, args
        return plan.heat_step(_raw(x), *args)

    @staticmethod
    def backward(ctx, g):
        return (ctx.plan.heat_step(_raw(g), *ctx.args),) + (None,) * (1 + len(ctx.args))


class _SolveMisfit(torch.autograd.Function):
    @staticmethod
    def forward(ctx, x, g, plan, *args):
        ctx.plan, ctx.args = plan, args
        r = plan.spectral_solve(_raw(x), *args)
        loss = plan.residual_norm(r, g)
        ctx.save_for_backward(r)
        return loss

    @staticmethod
    def backward(ctx, gloss):
        (r,) = ctx.saved_tensors
        grad = ctx.plan.spectral_solve(_raw(r), *ctx.args, adjoint=True, factor=2.0 * gloss.to(torch.float64))
        return (grad,) + (None,) * (2 + len(ctx.args))


def fft(x, plan):
    """forward_fft: real-space packed layout -> reciprocal layout."""
    return _Forward.apply(x, plan)


def ifft(x, plan, scale=None):
    """inverse_fft with `scale` (default 1/N^d)."""
    if scale is None:
        scale = 1.0 / float(plan.shape.n) ** plan.shape.dims
    return _Inverse.apply(x, plan, float(scale))


def laplace(x, plan, scale=1.0):
    return _Laplace.apply(x, plan, float(scale))


def dx4(x, plan, delta=1.0):
    return _Dx4.apply(x, plan, float(delta))


def dy4(x, plan, delta=1.0):
    return _Dy4.apply(x, plan, float(delta))


def dz4(x, plan, delta=1.0):
    return _Dz4.apply(x, plan, float(delta))


def spectral(x, plan, kind, p0=0.0, p1=0.0, length=1.0):
    return _Spectral.apply(x, plan, kind, float(p0), float(p1), float(length))


def spectral_solve(x, plan, kind, p0=0.0, p1=0.0, length=1.0, scale=None):
    """ifft(spectral(fft(x))) with `scale` (default 1/N^d) as one operator."""
    if scale is None:
        scale = 1.0 / float(plan.shape.n) ** plan.shape.dims
    return _SpectralSolve.apply(x, plan, kind, float(p0), float(p1), float(length), float(scale))


def heat_step(x, plan, nu, dt, lap_scale=1.0, length=1.0):
    """ifft(exp(-nu |k|^2 dt) fft(x)) + dt laplace(x, lap_scale) as one operator."""
    return _HeatStep.apply(x, plan, float(nu), float(dt), float(lap_scale), float(length))


def solve_misfit(x, g, plan, kind, p0=0.0, p1=0.0, length=1.0):
    """||spectral_solve(x) - g||^2, differentiable in x; g is a constant."""
    scale = 1.0 / float(plan.shape.n) ** plan.shape.dims
    return _SolveMisfit.apply(x, g, plan, kind, float(p0), float(p1), float(length), scale)
