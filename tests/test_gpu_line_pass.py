"""The natural-order line passes against numpy-order FFTs in FP64 (torch on the
GPU), through zm_forward / zm_inverse: every line length they are built for, the
fewest and most ranks, the smallest and largest blocks and vectors, odd batches
(one field takes the passes' small variants, several the large ones).

Bars: FP64 within 1e-13 relative max error; FP32 within 1e-6 relative L2 and
1e-5 relative max, those of every transform test here."""
import sys

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

# (dims, N, P, B, batch); VEC = N / (P B) >= P
SHAPES = [(2, 16, 1, 2, 3), (2, 16, 4, 1, 1), (2, 32, 2, 2, 1), (2, 32, 4, 2, 7), (2, 64, 8, 1, 1), (2, 64, 1, 64, 3),
          (2, 128, 8, 2, 1), (2, 128, 2, 2, 67), (2, 256, 4, 16, 1), (2, 256, 1, 2, 17), (2, 512, 8, 8, 1),
          (2, 512, 2, 64, 5), (2, 1024, 1, 4, 1), (2, 1024, 8, 16, 5), (2, 2048, 8, 32, 1), (2, 2048, 1, 2, 3),
          (2, 4096, 1, 4, 1), (2, 4096, 16, 16, 1), (2, 8192, 2, 8, 1), (3, 16, 4, 1, 1), (3, 16, 1, 16, 3),
          (3, 32, 2, 8, 1), (3, 32, 4, 1, 5), (3, 64, 8, 1, 1), (3, 64, 1, 2, 1), (3, 128, 4, 8, 1), (3, 128, 2, 1, 2),
          (3, 256, 8, 2, 1), (3, 256, 2, 64, 1), (3, 512, 4, 2, 1)]


def _pack(x, dims, n, p, b):
    vec = n // (p * b)
    if dims == 2:
        t = x.reshape(-1, vec, p, b, vec, p, b).permute(0, 2, 5, 1, 3, 6, 4)
    else:
        t = x.reshape(-1, vec, p, b, vec, p, b, vec, p, b).permute(0, 2, 5, 8, 1, 3, 4, 6, 9, 7)
    return t.reshape(-1).contiguous()


def _reciprocal(s, dims, n, p, b):
    m, vp = p * b, n // (p * p * b)
    if dims == 2:
        t = s.reshape(-1, m, p, vp, m, p, vp).permute(0, 2, 5, 4, 6, 1, 3)
    else:
        t = s.reshape(-1, m, p, vp, m, p, vp, m, p, vp).permute(0, 2, 5, 8, 4, 6, 7, 9, 1, 3)
    return t.reshape(-1).contiguous()


def _errors(a, ref):
    d = (a.to(torch.complex128) - ref).abs()
    return ((torch.linalg.vector_norm(d) / torch.linalg.vector_norm(ref)).item(),
            (d.max() / ref.abs().max()).item())


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims,n,p,b,batch", SHAPES)
def test_transforms_against_fft(dims, n, p, b, batch, precision):
    from stencilfft_amd import Plan
    print(f"[gpu] line pass {precision} {dims}D N={n} P={p} B={b} batch {batch}", flush=True)
    sys.stdout.flush()
    pl = Plan(dims, n, p, b, precision=precision, batch=batch)
    g = torch.Generator(device="cuda")
    g.manual_seed(n + 7 * p + b)
    parts = torch.rand((batch,) + (n,) * dims + (2,), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    x = torch.view_as_complex(parts).to(pl.complex_dtype)
    axes = tuple(range(1, dims + 1))
    spec = torch.fft.fftn(x.to(torch.complex128), dim=axes)
    want = _reciprocal(spec, dims, n, p, b)
    packed = _pack(x, dims, n, p, b)
    keep = packed.clone()
    y = pl.forward(packed)
    l2, mx = _errors(y, want)
    # the inverse from the rounded spectrum: its own error alone
    yin = want.to(pl.complex_dtype)
    z = pl.inverse(yin, 1.0 / float(n) ** dims)
    back = _pack(x.to(torch.complex128), dims, n, p, b)
    zl2, zmx = _errors(z, back)
    assert torch.equal(packed, keep)
    if precision == "fp64":
        assert mx < 1e-13 and zmx < 1e-13, (mx, zmx)
    else:
        assert l2 < 1e-6 and mx < 1e-5 and zl2 < 1e-6 and zmx < 1e-5, (l2, mx, zl2, zmx)


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims,n,p,b,batch", [s for s in SHAPES if s[1] <= 2048] + [(3, 32, 1, 1, 2), (2, 64, 2, 1, 3)])
def test_laplace_forward_bits(dims, n, p, b, batch, precision):
    """The Laplacian formed in the x pass: bit for bit the two calls, at the wrap
    of rows, planes and columns, in blocks of one and across every rank edge."""
    from stencilfft_amd import Plan
    print(f"[gpu] laplace + line pass {precision} {dims}D N={n} P={p} B={b} batch {batch}", flush=True)
    sys.stdout.flush()
    pl = Plan(dims, n, p, b, precision=precision, batch=batch)
    g = torch.Generator(device="cuda")
    g.manual_seed(3 * n + p)
    parts = torch.rand((pl.numel(), 2), generator=g, device="cuda", dtype=torch.float64) * 2 - 1
    x = torch.view_as_complex(parts).to(pl.complex_dtype)
    for scale in (1.0, float(n * n)):
        want = torch.view_as_real(pl.forward(pl.laplace(x, scale))).view(torch.int8)
        got = torch.view_as_real(pl.laplace_forward(x, scale)).view(torch.int8)
        assert torch.equal(got, want)
