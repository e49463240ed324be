"""zm_spectral_solve against its three calls (zm_forward, zm_spectral_multiply,
zm_inverse) in FP64, for every multiplier and both plans' paths (tiles, rows at
N >= 4096, generic fallback, MFMA, two-stage), and its adjoint identity.

Bars: both sides round the same chain, so FP64 agrees within the transforms' own
1e-13 relative max and FP32 within 1e-6 relative L2 of the FP64 chain."""
import sys

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

KINDS = [("poisson", 0.0, 0.0), ("heat", 1e-3, 1e-2), ("scale", 1.5, 0.0), ("stencil", 2.0, 0.0),
         ("poisson_stencil", 2.0, 0.0)]
KINDS_2D = [("stencil", 2.0, 0.25), ("poisson_stencil", 2.0, 0.25)]
# (dims, N, P, B, batch)
SHAPES = [(2, 8, 2, 1, 1), (2, 16, 4, 1, 3), (2, 32, 2, 2, 1), (2, 64, 4, 2, 1), (2, 128, 8, 2, 5), (2, 256, 2, 8, 2),
          (2, 256, 4, 8, 40), (2, 512, 8, 8, 1), (2, 1024, 2, 16, 1), (2, 1024, 1, 4, 5), (2, 2048, 4, 16, 1),
          (2, 4096, 4, 16, 1), (2, 4096, 8, 2, 1), (2, 8192, 2, 32, 1), (3, 16, 2, 2, 1), (3, 32, 4, 1, 3),
          (3, 64, 2, 4, 1), (3, 128, 4, 8, 1), (3, 256, 2, 8, 1)]


def _field(pl, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    parts = torch.rand((pl.numel(), 2), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    return torch.view_as_complex(parts).to(pl.complex_dtype)


def _rel(a, ref):
    d = (a.to(torch.complex128) - ref).abs()
    return ((torch.linalg.vector_norm(d) / torch.linalg.vector_norm(ref)).item(),
            (d.max() / ref.abs().max()).item())


@pytest.mark.parametrize("dims,n,p,b,batch", SHAPES)
def test_solve_is_the_three_calls(dims, n, p, b, batch):
    from stencilfft_amd import Plan
    print(f"[gpu] spectral solve {dims}D N={n} P={p} B={b} batch {batch}", flush=True)
    sys.stdout.flush()
    p64 = Plan(dims, n, p, b, precision="fp64", batch=batch)
    x = _field(p64, n + p)
    p32 = Plan(dims, n, p, b, precision="fp32", batch=batch)
    x32 = x.to(torch.complex64)
    scale = 1.0 / float(n) ** dims
    for kind, a0, a1 in KINDS + (KINDS_2D if dims == 2 else []):
        for adjoint in (False, True):
            def calls(u):
                y = p64.forward(u)
                p64.spectral_multiply(y, kind, a0, a1, out=y, adjoint=adjoint)
                return p64.inverse(y, scale)
            want = calls(x)
            keep = x.clone()
            got = p64.spectral_solve(x, kind, a0, a1, scale=scale, adjoint=adjoint)
            assert _rel(got, want)[1] < 1e-13, (kind, a1, adjoint)
            assert torch.equal(x, keep)
            got32 = p32.spectral_solve(x32, kind, a0, a1, scale=scale, adjoint=adjoint)
            assert _rel(got32, calls(x32.to(torch.complex128)))[0] < 1e-6, (kind, a1, adjoint)


@pytest.mark.parametrize("precision,two_stage", [("fp32_mfma", False), ("fp64", True)])
def test_fallback_paths(precision, two_stage):
    from stencilfft_amd import Plan
    print(f"[gpu] spectral solve fallback {precision}", flush=True)
    pl = Plan(2, 256, 2, 8, precision=precision, two_stage=two_stage)
    x = _field(pl, 3)
    y = pl.forward(x)
    pl.spectral_multiply(y, "heat", 1e-3, 1e-2, out=y)
    want = pl.inverse(y, 0.5)
    assert torch.equal(pl.spectral_solve(x, "heat", 1e-3, 1e-2, scale=0.5), want)
    two = torch.full((), 2.0, dtype=torch.float64, device="cuda")  # a power of two scales exactly
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    for stream in (None, side):
        got = pl.spectral_solve(x, "heat", 1e-3, 1e-2, scale=0.5, factor=two, stream=stream)
        torch.cuda.synchronize()
        assert torch.equal(got, 2 * want)


def test_arguments_are_checked_before_any_launch():
    import ctypes
    from stencilfft_amd import Plan, ZmError
    from stencilfft_amd import _lib as L
    print("[gpu] spectral solve arguments", flush=True)
    pl = Plan(3, 16, 2, 2, precision="fp64")
    x, out = _field(pl, 1), torch.full((pl.numel(),), 7.0, dtype=torch.complex128, device="cuda")
    for kw in (dict(kind="stencil", p1=0.5), dict(kind="heat", length=0.0)):
        with pytest.raises(ZmError) as e:
            pl.spectral_solve(x, out=out, **kw)
        assert e.value.status == L.ZM_ERR_INVALID_ARG
    fn = L._lib().zm_spectral_solve
    ptr = ctypes.c_void_p(x.data_ptr())
    assert fn(pl.handle, ptr, ptr, 0, 0.0, 0.0, 1.0, 1.0, None, None, None) == L.ZM_ERR_ALIAS
    assert fn(pl.handle, ptr, out.data_ptr(), 0, 0.0, 0.0, 1.0, 1.0, None, ptr, None) == L.ZM_ERR_ALIAS
    assert fn(pl.handle, ptr, out.data_ptr(), 9, 0.0, 0.0, 1.0, 1.0, None, None, None) == L.ZM_ERR_INVALID_ARG
    two = Plan(2, 256, 2, 8, precision="fp64", two_stage=True)
    a, b = _field(two, 1), _field(two, 2)
    assert fn(two.handle, a.data_ptr(), b.data_ptr(), 0, 0.0, 0.0, 1.0, 1.0, None, None, None) == L.ZM_ERR_UNSUPPORTED
    torch.cuda.synchronize()
    assert bool((out == 7.0).all())


@pytest.mark.parametrize("dims,n,p,b,batch", [(2, 64, 4, 2, 3), (2, 1024, 2, 16, 1), (2, 4096, 4, 16, 1), (3, 16, 2, 2, 1),
                                              (3, 64, 2, 4, 2), (3, 128, 4, 2, 1), (3, 256, 1, 64, 1)])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_heat_step_is_solve_plus_laplacian(dims, n, p, b, batch, precision):
    """The accumulating Laplacian (generic, strip and march kernels) rounds like
    the separate product and sum, so the step is bit for bit their result."""
    from stencilfft_amd import Plan, solvers
    print(f"[gpu] heat step {precision} {dims}D N={n} P={p} B={b} batch {batch}", flush=True)
    pl = Plan(dims, n, p, b, precision=precision, batch=batch)
    x = _field(pl, n)
    u = pl.spectral_solve(x, "heat", 1e-3, 0.03, 1.0, 1.0 / float(n) ** dims)
    want = u + 0.03 * pl.laplace(x, 1.5)
    assert torch.equal(solvers.heat_step(x, pl, 1e-3, 0.03, lap_scale=1.5), want)
    g = _field(pl, n + 1)
    xr = x.clone().requires_grad_(True)
    (grad,) = torch.autograd.grad(solvers.heat_step(xr, pl, 1e-3, 0.03, lap_scale=1.5), xr, grad_outputs=g)
    assert torch.equal(grad, solvers.heat_step(g, pl, 1e-3, 0.03, lap_scale=1.5))
    # a tensor time step takes the operators one by one
    dt = torch.full((), 0.03, dtype=pl.real_dtype, device="cuda")
    assert _rel(solvers.heat_step(x, pl, 1e-3, dt, lap_scale=1.5), want.to(torch.complex128))[1] < 1e-5


@pytest.mark.parametrize("n,p,b,batch,precision,two_stage", [
    (16, 2, 2, 1, "fp64", False), (64, 4, 2, 3, "fp32", False), (512, 2, 16, 3, "fp64", False),
    (2048, 4, 16, 1, "fp32", False), (4096, 4, 16, 1, "fp32", False), (256, 2, 8, 2, "fp64", True)])
def test_poisson_misfit_and_its_gradient(n, p, b, batch, precision, two_stage):
    """The fused loss against ||residual||^2 by torch in FP64 on the same
    residual, and its gradient (an incoming gradient of 3 included) against the
    chain with a target that needs a gradient, which runs the operators apart."""
    from stencilfft_amd import Plan, solvers
    print(f"[gpu] poisson misfit {precision} N={n} P={p} B={b} batch {batch}", flush=True)
    pl = Plan(2, n, p, b, precision=precision, batch=batch, two_stage=two_stage)
    eps = torch.finfo(pl.real_dtype).eps
    f, g = _field(pl, 1).requires_grad_(True), _field(pl, 2)
    loss = solvers.poisson_loss(f, g, pl, form="spectral")
    r = solvers.poisson_residual(f.detach(), g, pl, form="spectral").to(torch.complex128)
    ref = torch.view_as_real(r).pow(2).sum()
    assert loss.shape == () and loss.dtype == pl.real_dtype
    assert abs(loss.item() - ref.item()) <= (4 * eps if precision == "fp32" else 1e-13) * ref.item()
    (grad,) = torch.autograd.grad(3.0 * loss, f)
    gg = g.clone().requires_grad_(True)
    want_f, want_g = torch.autograd.grad(3.0 * solvers.poisson_loss(f, gg, pl, form="spectral"), (f, gg))
    assert _rel(grad, want_f.to(torch.complex128))[0] < 8 * eps
    assert _rel(want_g, -6.0 * r)[0] < 8 * eps
    # strided input, and a loss that needs no gradient
    wide = torch.stack([f.detach(), g], dim=1)[:, 0]
    assert solvers.poisson_loss(wide, g, pl, form="spectral").item() == loss.item()
