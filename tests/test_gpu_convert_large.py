"""The layout converters on fields that the last-level cache cannot hold (256 MB),
which take non-temporal loads, and on fields of the cache's size: bit for bit the
permutation, both ways, with tiles within a row, of rows, and of planes."""
import sys

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_line_pass import _pack  # noqa: E402

# (dims, N, P, B, batch, precision): 256 MB, then larger
SHAPES = [(2, 4096, 4, 16, 1, "fp64"), (2, 4096, 2, 64, 2, "fp32"), (2, 4096, 8, 4, 2, "fp64"),
          (2, 8192, 4, 32, 1, "fp32"), (2, 32, 2, 4, 20000, "fp64"), (3, 256, 2, 8, 3, "fp32"), (3, 32, 4, 1, 600, "fp64"),
          (2, 16, 1, 4, 65535, "fp64")]


@pytest.mark.parametrize("dims,n,p,b,batch,precision", SHAPES)
def test_converters_beyond_the_cache(dims, n, p, b, batch, precision):
    from stencilfft_amd import Plan
    print(f"[gpu] convert {precision} {dims}D N={n} P={p} B={b} batch {batch}", flush=True)
    sys.stdout.flush()
    pl = Plan(dims, n, p, b, precision=precision, batch=batch, caller_scratch=True)
    k = torch.arange(pl.numel(), dtype=pl.real_dtype, device="cuda")  # exact in FP32 up to 2^24
    x = torch.complex(k % (1 << 24), k // (1 << 24))
    want = _pack(x.reshape((batch,) + (n,) * dims), dims, n, p, b)
    packed = pl.natural_to_packed(x)
    assert torch.equal(packed, want)
    assert torch.equal(pl.packed_to_natural(packed), x)
