"""The derivative and depth marches on fields too small for their wide shapes
(single lines, strips down to 8 positions, 4 planes) and on either side of that
rule: all fields of a batch against periodic differences in FP64 (torch.roll in
natural order).  Each value is four products and sums (the Laplacian six sums),
so FP64 agrees within 16 eps of the largest term and FP32, on FP32 input, within
16 of its own."""
import sys

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# (dims, N, P, B, batch)
SHAPES = [(2, 16, 2, 2, 1), (2, 256, 4, 8, 3), (2, 1024, 2, 16, 1), (2, 1024, 8, 4, 2), (2, 2048, 1, 32, 1),
          (2, 4096, 4, 16, 1), (3, 16, 1, 4, 1), (3, 32, 2, 2, 5), (3, 64, 4, 2, 1), (3, 128, 2, 16, 1),
          (3, 128, 1, 8, 2), (3, 256, 4, 8, 1)]


def _pack(x, dims, n, p, b):
    vec = n // (p * b)
    if dims == 2:
        t = x.reshape(-1, vec, p, b, vec, p, b).permute(0, 2, 5, 1, 3, 6, 4)
    else:
        t = x.reshape(-1, vec, p, b, vec, p, b, vec, p, b).permute(0, 2, 5, 8, 1, 3, 4, 6, 9, 7)
    return t.reshape(-1).contiguous()


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims,n,p,b,batch", SHAPES)
def test_marches_against_differences(dims, n, p, b, batch, precision):
    from stencilfft_amd import Plan
    print(f"[gpu] marches {precision} {dims}D N={n} P={p} B={b} batch {batch}", flush=True)
    sys.stdout.flush()
    pl = Plan(dims, n, p, b, precision=precision, batch=batch)
    g = torch.Generator(device="cuda")
    g.manual_seed(n + b)
    u = torch.rand((batch,) + (n,) * dims, generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    for x in (u.to(pl.real_dtype), torch.complex(u, u.flip(1)).to(pl.complex_dtype)):
        nat = x.to(torch.complex128 if x.is_complex() else torch.float64)
        packed = _pack(x, dims, n, p, b)
        tol = 16 * torch.finfo(pl.real_dtype).eps
        for axis, fn in ((dims, pl.dx4), (dims - 1, pl.dy4), (dims - 2, pl.dz4 if dims == 3 else None)):
            if fn is None:
                continue
            want = (8 * (torch.roll(nat, -1, axis) - torch.roll(nat, 1, axis))
                    - (torch.roll(nat, -2, axis) - torch.roll(nat, 2, axis))) / (12 * 0.5)
            got = fn(packed, 0.5).to(nat.dtype)
            assert (got - _pack(want, dims, n, p, b)).abs().max().item() < tol * 8 * 2 / 6, fn.__name__
        want = sum(torch.roll(nat, s, a) for a in range(1, dims + 1) for s in (1, -1)) - 2 * dims * nat
        got = pl.laplace(packed, 1.0).to(nat.dtype)
        assert (got - _pack(want, dims, n, p, b)).abs().max().item() < tol * 2 * 2 * dims


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("n,p,b,batch", [(64, 2, 4, 8), (64, 1, 4, 16), (128, 2, 8, 8), (128, 4, 4, 8), (256, 2, 8, 3),
                                         (256, 1, 16, 1)])
def test_depth_strips_leave_every_value(n, p, b, batch, precision):
    """A batch's depth strips are as long as its size asks for; each value is
    the same sum whatever the strip, so the batch equals its fields alone bit
    for bit, and the accumulating form equals the two operations."""
    from stencilfft_amd import Plan
    print(f"[gpu] depth strips {precision} N={n} P={p} B={b} batch {batch}", flush=True)
    sys.stdout.flush()
    pl, one = Plan(3, n, p, b, precision=precision, batch=batch), Plan(3, n, p, b, precision=precision)
    g = torch.Generator(device="cuda")
    g.manual_seed(n + batch)
    x, z = (torch.rand((2, pl.numel()), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
            ).to(pl.real_dtype).repeat_interleave(2, 1).reshape(2, -1, 2).unbind(0)
    x, z = torch.view_as_complex(x.contiguous()), torch.view_as_complex((z * 0.5).contiguous())
    lap = pl.laplace(x, 2.0)
    for xf, lf in zip(x.chunk(batch), lap.chunk(batch)):
        assert torch.equal(one.laplace(xf.contiguous(), 2.0), lf)
    want = torch.view_as_real(z) + 0.25 * torch.view_as_real(lap)
    assert torch.equal(torch.view_as_real(pl.laplace_add(x, z, 2.0, 0.25)), want)
