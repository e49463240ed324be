"""Either side of the sizes at which the FP64 marches shorten their strips and the
FP64 converter takes other stores: a batch takes one side, its fields alone the
other.  The values do not depend on the side, so they agree bit for bit."""
import sys

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_line_pass import _pack  # noqa: E402


def _fields(pl, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.view_as_complex(torch.rand((pl.numel(), 2), generator=g, device="cuda", dtype=torch.float64) * 2 - 1)


# workgroups of a field: y lines of 64 in 32, of 128 in 256; depth tiles of L = 64
# in 16 (N = 64), 64 (N = 128) and 128 (N = 256) per strip
@pytest.mark.parametrize("n,p,b,batch", [(64, 2, 4, 16), (64, 1, 8, 5), (128, 4, 2, 2), (128, 2, 4, 8), (256, 4, 16, 3)])
def test_fp64_strips_leave_every_value(n, p, b, batch):
    from stencilfft_amd import Plan
    print(f"[gpu] FP64 strips N={n} P={p} B={b} batch {batch}", flush=True)
    sys.stdout.flush()
    one, pl = (Plan(3, n, p, b, precision="fp64", batch=k, caller_scratch=True) for k in (1, batch))
    x, acc = _fields(pl, n), _fields(pl, n + 1)
    for fn in (lambda q, u, a: q.dy4(u, 0.5), lambda q, u, a: q.laplace(u, 1.5),
               lambda q, u, a: q.laplace_add(u, a.clone(), 1.5, 0.25)):
        want = torch.cat([fn(one, u, a) for u, a in zip(x.chunk(batch), acc.chunk(batch))])
        assert torch.equal(fn(pl, x, acc), want)


# rank rows of 64 bytes (of 128 in the third): the last batch of 128 MB, and the
# first beyond it
@pytest.mark.parametrize("dims,n,p,b,batch", [(3, 16, 4, 1, 2048), (3, 16, 4, 1, 2049), (3, 16, 2, 1, 2048),
                                              (3, 8, 2, 1, 16384), (3, 8, 2, 1, 16385), (2, 64, 1, 4, 2048)])
def test_converter_stores_on_either_side(dims, n, p, b, batch):
    from stencilfft_amd import Plan
    print(f"[gpu] convert {dims}D N={n} P={p} B={b} batch {batch}", flush=True)
    sys.stdout.flush()
    pl = Plan(dims, n, p, b, precision="fp64", batch=batch, caller_scratch=True)
    x = _fields(pl, batch)
    packed = pl.natural_to_packed(x)
    assert torch.equal(packed, _pack(x.reshape((batch,) + (n,) * dims), dims, n, p, b))
    assert torch.equal(pl.packed_to_natural(packed), x)
