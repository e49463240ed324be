"""Either side of the sizes at which the FP64 marches shorten their strips: a batch
takes one side, its fields alone the other.  The values do not depend on the side,
so they agree bit for bit."""
import sys

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def _fields(pl, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return torch.view_as_complex(torch.rand((pl.numel(), 2), generator=g, device="cuda", dtype=torch.float64) * 2 - 1)


# workgroups of a field: y lines of 64 in 32, of 128 in 256
@pytest.mark.parametrize("n,p,b,batch", [(64, 2, 4, 16), (64, 1, 8, 5), (128, 4, 2, 2), (128, 2, 4, 8), (256, 4, 16, 3)])
def test_fp64_strips_leave_every_value(n, p, b, batch):
    from stencilfft_amd import Plan
    print(f"[gpu] FP64 strips N={n} P={p} B={b} batch {batch}", flush=True)
    sys.stdout.flush()
    one, pl = (Plan(3, n, p, b, precision="fp64", batch=k, caller_scratch=True) for k in (1, batch))
    x = _fields(pl, n)
    want = torch.cat([one.dy4(u, 0.5) for u in x.chunk(batch)])
    assert torch.equal(pl.dy4(x, 0.5), want)
