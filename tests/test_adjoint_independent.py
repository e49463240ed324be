"""adjoint_heat as a check on the fused heat step: it runs the operators one by
one (on the CPU against a stand-in plan that has only those), and on the GPU the
fused operators' gradients hold against it and against finite differences."""
import sys

import pytest

torch = pytest.importorskip("torch")

from conftest import has_gpu  # noqa: E402

gpu = [pytest.mark.gpu, pytest.mark.skipif(not has_gpu(), reason="needs a GPU")]


class SeparateOperators:
    """Natural-order 2D operators on the CPU; no solve, step or accumulation."""

    def __init__(self, n):
        from stencilfft_amd import Shape
        self.shape = Shape(2, n, 1, 2)

    def _f(self, x):
        return x.reshape(self.shape.n, self.shape.n)

    def inverse_adjoint(self, x, scale):
        return scale * torch.fft.fft2(self._f(x)).reshape(-1)

    def forward_adjoint(self, x):
        return torch.fft.ifft2(self._f(x), norm="forward").reshape(-1)

    def decay(self, nu, dt, length):
        n = self.shape.n
        k = torch.fft.fftfreq(n, 1.0 / n, dtype=torch.float64) * (2 * torch.pi / length)
        return torch.exp(-nu * (k[:, None] ** 2 + k ** 2) * dt)

    def spectral_multiply(self, x, kind, nu, dt, length, adjoint):
        assert kind == "heat" and adjoint
        return (self._f(x) * self.decay(nu, dt, length)).reshape(-1)

    def laplace(self, x, scale):
        f = self._f(x)
        return scale * (sum(torch.roll(f, s, d) for d in (0, 1) for s in (1, -1)) - 4 * f).reshape(-1)


def test_adjoint_heat_runs_the_operators_apart():
    from stencilfft_amd import solvers
    n, nu, dt, lap = 16, 1e-3, 1e-2, 1.5
    pl = SeparateOperators(n)
    gen = torch.Generator()
    gen.manual_seed(1)
    g = torch.randn(n * n, dtype=torch.complex128, generator=gen)
    got = solvers.adjoint_heat(g, pl, 3, nu, dt, lap_scale=lap)
    want = g  # the step is real and symmetric in Fourier space
    for _ in range(3):
        smooth = torch.fft.ifft2(torch.fft.fft2(pl._f(want)) * pl.decay(nu, dt, 1.0)).reshape(-1)
        want = smooth + dt * pl.laplace(want, lap)
    assert (got - want).abs().max().item() <= 1e-13 * want.abs().max().item()


@pytest.mark.parametrize("dims,n,p,b", [pytest.param(*s, marks=gpu) for s in [(2, 16, 2, 2), (3, 8, 2, 1), (3, 16, 2, 2)]])
def test_gradcheck_of_the_fused_operators(dims, n, p, b):
    from stencilfft_amd import Plan
    from stencilfft_amd import autograd as ag
    from helpers import uniform_field
    print(f"[gpu] gradcheck of solve, step and misfit {dims}D N={n}", flush=True)
    sys.stdout.flush()
    pl = Plan(dims, n, p, b, precision="fp64")
    x, t = (torch.from_numpy(uniform_field(pl.numel(), s)).cuda() for s in (1, 2))
    x.requires_grad_(True)
    dx = 0.25 if dims == 2 else 0.0
    for op in (lambda u: ag.spectral_solve(u, pl, "heat", 0.01, 0.5), lambda u: ag.spectral_solve(u, pl, "poisson"),
               lambda u: ag.spectral_solve(u, pl, "poisson_stencil", 2.0, dx, scale=0.5),
               lambda u: ag.heat_step(u, pl, 0.01, 0.05, 1.5),
               lambda u: ag.solve_misfit(u, t, pl, "poisson_stencil", 2.0, dx)):
        # linear or quadratic: central differences are exact at any eps, so a
        # large one leaves the rounding of losses of up to 1e4 below 1e-9
        assert torch.autograd.gradcheck(op, (x,), eps=1e-3, atol=1e-8, rtol=1e-6, fast_mode=True)


@pytest.mark.parametrize("dims,n,p,b,precision", [pytest.param(*s, marks=gpu) for s in [
    (2, 64, 4, 2, "fp64"), (2, 4096, 4, 16, "fp32"), (3, 32, 2, 2, "fp64"), (3, 64, 2, 4, "fp32"), (3, 256, 4, 4, "fp64")]])
def test_fused_step_against_the_operators_apart(dims, n, p, b, precision):
    """Four steps forward and back through the fused step, and the same gradient
    through the separate operators: each transform pair rounds at the level of
    the transform tests' bars (1e-13 relative max in FP64, 1e-6 relative L2 in
    FP32)."""
    from stencilfft_amd import Plan, solvers
    print(f"[gpu] fused heat step {precision} {dims}D N={n}", flush=True)
    sys.stdout.flush()
    pl = Plan(dims, n, p, b, precision=precision)
    gen = torch.Generator(device="cuda")
    gen.manual_seed(n)
    g, u0 = (torch.view_as_complex(torch.rand((pl.numel(), 2), generator=gen, device="cuda",
                                              dtype=torch.float64) * 2 - 1).to(pl.complex_dtype) for _ in range(2))
    u0.requires_grad_(True)
    u = u0
    for _ in range(4):
        u = solvers.heat_step(u, pl, 1e-3, 1e-2)
    (got,) = torch.autograd.grad(u, u0, grad_outputs=g)
    want = solvers.adjoint_heat(g, pl, 4, 1e-3, 1e-2)
    d = (got - want).to(torch.complex128)
    if precision == "fp64":
        assert (d.abs().max() / want.abs().max()).item() < 4e-13
    else:
        assert (torch.linalg.vector_norm(d) / torch.linalg.vector_norm(want)).item() < 4e-6
