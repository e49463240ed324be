"""natural <-> packed conversion, bit for bit, at tile edges: fields smaller than
a tile, single-column and single-row splits (VEC = 1, M = 1), blocks and vectors
longer than a tile, batches; both precisions and directions."""
import sys

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

SHAPES = [(2, 16, 1, 16, 1), (2, 16, 4, 1, 3), (2, 32, 1, 1, 2), (2, 64, 8, 1, 5), (2, 64, 1, 64, 1), (2, 256, 2, 64, 1),
          (2, 1024, 1, 1, 1), (2, 1024, 1, 1024, 1), (2, 2048, 8, 4, 3), (2, 4096, 2, 1024, 1), (2, 8192, 4, 2, 1),
          (3, 8, 2, 1, 1), (3, 16, 4, 1, 2), (3, 32, 1, 32, 1), (3, 64, 2, 2, 1), (3, 128, 4, 8, 1), (3, 256, 1, 1, 1)]


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("dims,n,p,b,batch", SHAPES)
def test_conversion_is_the_permutation(dims, n, p, b, batch, precision):
    from stencilfft_amd import Plan
    print(f"[gpu] convert {precision} {dims}D N={n} P={p} B={b} batch {batch}", flush=True)
    sys.stdout.flush()
    pl = Plan(dims, n, p, b, precision=precision, batch=batch)
    vec = n // (p * b)
    re = torch.arange(pl.numel(), device="cuda", dtype=torch.float64)
    x = torch.complex(re, -re - 1).to(pl.complex_dtype)
    if dims == 2:
        t = x.reshape(-1, vec, p, b, vec, p, b).permute(0, 2, 5, 1, 3, 6, 4)
    else:
        t = x.reshape(-1, vec, p, b, vec, p, b, vec, p, b).permute(0, 2, 5, 8, 1, 3, 4, 6, 9, 7)
    want = t.reshape(-1).contiguous()
    got = pl.natural_to_packed(x)
    assert torch.equal(torch.view_as_real(got), torch.view_as_real(want))
    assert torch.equal(torch.view_as_real(pl.packed_to_natural(got)), torch.view_as_real(x))
