"""Tensors whose storage is not their value: lazily conjugated or negated, a
subclass that computes its values, or with a forward-mode tangent.  The library
reads storage, so the operators carry lazy forms out first, and a Poisson target
of any of these forms takes the separate operators, as torch evaluates them.

On the CPU a stand-in plan reads storage through data_ptr() like the library's
entries do; on the GPU the plan itself."""
import ctypes
import sys

import numpy as np
import pytest

torch = pytest.importorskip("torch")

from conftest import has_gpu  # noqa: E402

SHAPE = (2, 16, 2, 2)


class RawPlan:
    """The plan's operators on CPU fields in natural order, from raw storage."""

    complex_dtype, real_dtype = torch.complex128, torch.float64

    def __init__(self):
        from stencilfft_amd import Shape
        self.shape = Shape(*SHAPE)

    @staticmethod
    def raw(t):
        nbytes = t.numel() * t.element_size()
        buf = (ctypes.c_char * nbytes).from_address(t.data_ptr())
        return torch.from_numpy(np.frombuffer(buf, dtype=np.complex128).copy())

    def spectral_solve(self, x, kind, p0, p1, length, scale, adjoint=False, factor=None):
        n = self.shape.n
        k = torch.arange(n * n, dtype=torch.float64).reshape(n, n)
        m = torch.polar(1 / (1 + k), 0.1 * k)
        m = m.conj() if adjoint else m
        if factor is not None:
            m = m * factor
        return (torch.fft.ifft2(m * torch.fft.fft2(self.raw(x).reshape(n, n)))).reshape(x.shape)

    def heat_step(self, x, nu, dt, lap_scale, length):
        return 3.0 * self.raw(x).reshape(x.shape)

    def residual_norm(self, acc, g):
        acc.copy_(self.raw(acc) - self.raw(g))
        return torch.view_as_real(acc).pow(2).sum()


def _fields(device):
    gen = torch.Generator()
    gen.manual_seed(5)
    return [torch.randn(SHAPE[1] ** 2, dtype=torch.complex128, generator=gen).to(device) for _ in range(2)]


def _plan(device):
    if device == "cpu":
        return RawPlan()
    from stencilfft_amd import Plan
    return Plan(*SHAPE, precision="fp64")


DEVICES = ["cpu", pytest.param("cuda", marks=[pytest.mark.gpu, pytest.mark.skipif(not has_gpu(), reason="needs a GPU")])]


class Doubled(torch.Tensor):
    """Twice its storage in every operation."""

    @classmethod
    def __torch_function__(cls, func, types, args=(), kwargs=None):
        plain = [a.as_subclass(torch.Tensor) for a in args if type(a) is cls]
        if func in (torch.Tensor.sub, torch.Tensor.__rsub__, torch.sub, torch.Tensor.add):
            args = [2 * plain.pop(0) if type(a) is cls else a for a in args]
            return func(*args, **(kwargs or {}))
        return super().__torch_function__(func, types, args, kwargs)


FORMS = {"conj": (torch.Tensor.conj, torch.conj_physical), "neg": (torch._neg_view, torch.Tensor.neg),
         "neg_conj": (lambda t: torch._neg_view(t.conj()), lambda t: -torch.conj_physical(t)),
         "subclass": (lambda t: t.as_subclass(Doubled), lambda t: 2 * t)}


@pytest.mark.parametrize("device", DEVICES)
@pytest.mark.parametrize("form", FORMS)
def test_loss_of_a_target_that_is_not_its_storage(form, device):
    """Loss and gradient agree with those of the same target written out, to the
    rounding of 256 terms."""
    from stencilfft_amd import solvers
    print(f"target {form} on {device}", flush=True)
    sys.stdout.flush()
    pl = _plan(device)
    f, h = _fields(device)
    f.requires_grad_(True)
    lazy, written_out = FORMS[form]
    g, plain = lazy(h), written_out(h)
    got = solvers.poisson_loss(f, g, pl, form="spectral")
    want = solvers.poisson_loss(f, plain, pl, form="spectral")
    assert abs(got.item() - want.item()) <= 1e-13 * want.item()
    (gg,), (gw,) = torch.autograd.grad(got, f), torch.autograd.grad(want, f)
    assert (gg - gw).abs().max().item() <= 1e-12 * gw.abs().max().item()


@pytest.mark.parametrize("device", DEVICES)
def test_tangent_of_the_target(device):
    """Forward-mode differentiation along the target: d ||r||^2 = -2 Re <r, dg>."""
    from torch.autograd import forward_ad
    from stencilfft_amd import solvers
    print(f"target tangent on {device}", flush=True)
    pl = _plan(device)
    f, g = _fields(device)
    dg = f.flip(0).resolve_conj().clone()
    r = solvers.poisson_residual(f, g, pl, form="spectral")
    with forward_ad.dual_level():
        loss = solvers.poisson_loss(f, forward_ad.make_dual(g, dg), pl, form="spectral")
        got = forward_ad.unpack_dual(loss).tangent.item()
    want = -2 * torch.vdot(dg, r).real.item()
    scale = 2 * (torch.linalg.vector_norm(r) * torch.linalg.vector_norm(dg)).item()
    assert abs(got - want) <= 1e-13 * scale


def _operators(device):
    from stencilfft_amd import autograd as ag
    ops = {"spectral_solve": lambda t, pl: ag.spectral_solve(t, pl, "heat", 1e-3, 1e-2),
           "heat_step": lambda t, pl: ag.heat_step(t, pl, 1e-3, 1e-2),
           "solve_misfit": lambda t, pl: ag.solve_misfit(t, torch.ones_like(t, dtype=pl.complex_dtype), pl, "poisson")}
    if device == "cuda":
        ops.update({"fft": ag.fft, "ifft": ag.ifft, "laplace": ag.laplace, "dx4": ag.dx4, "dy4": ag.dy4,
                    "spectral": lambda t, pl: ag.spectral(t, pl, "stencil", 2.0, 0.25)})
    return ops


@pytest.mark.parametrize("device", DEVICES)
def test_operators_of_lazy_tensors(device):
    """Inputs and incoming gradients with the conjugation or negation still to be
    carried out: bit for bit the operator of the tensor written out."""
    pl = _plan(device)
    x, _ = _fields(device)
    for name, op in _operators(device).items():
        for form in ("conj", "neg", "neg_conj"):
            print(f"{name} of {form} on {device}", flush=True)
            lazy, written_out = FORMS[form]
            assert torch.equal(op(lazy(x), pl), op(written_out(x), pl)), (name, form)
            if name == "solve_misfit":  # a real loss
                continue
            xr = x.clone().requires_grad_(True)
            (got,) = torch.autograd.grad(op(xr, pl), xr, grad_outputs=lazy(x))
            (want,) = torch.autograd.grad(op(xr, pl), xr, grad_outputs=written_out(x))
            assert torch.equal(got, want), (name, form)


@pytest.mark.gpu
@pytest.mark.skipif(not has_gpu(), reason="needs a GPU")
def test_plan_refuses_lazy_tensors():
    pl = _plan("cuda")
    x, acc = _fields("cuda")
    factor = torch.ones((), dtype=torch.float64, device="cuda")
    for lazy in (x.conj(), torch._neg_view(x)):
        for call in (lambda: pl.spectral_solve(lazy, "poisson"), lambda: pl.spectral_solve(x, "poisson", out=lazy),
                     lambda: pl.heat_step(lazy, 1e-3, 1e-2), lambda: pl.laplace_add(lazy, acc),
                     lambda: pl.laplace_add(acc, lazy), lambda: pl.residual_norm(lazy, acc),
                     lambda: pl.residual_norm(acc, lazy)):
            with pytest.raises(ValueError, match="lazily"):
                call()
    with pytest.raises(ValueError, match="lazily"):
        pl.spectral_solve(x, "poisson", factor=torch._neg_view(factor))
