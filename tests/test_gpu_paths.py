"""What a plan runs, as zm_plan_path reports it and as the stage record shows it:
a fused path that fell back to its separate calls would still pass the tests of
its result, which compare it with those calls."""
import sys

import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_line_pass import SHAPES  # noqa: E402
from test_gpu_parity import SPECIALISED_PAIRS  # noqa: E402

PAIRS = [(2, v * m, 2, m // 2, 1) for v, m in SPECIALISED_PAIRS]


def _pair(n, p, b):
    return (n // (p * b), p * b) in SPECIALISED_PAIRS


# the split-precision variant takes the specialised pairs only
PLANS = [s + (prec,) for s in SHAPES + PAIRS + [(3, 1024, 2, 32, 1), (2, 64, 2, 2, 1), (2, 8, 2, 1, 1)]
         for prec in ("fp64", "fp32", "fp32_mfma") if prec != "fp32_mfma" or _pair(*s[1:4])]


def _expected(dims, n, p, b, precision):
    """(tiles, fused Laplacian, one-kernel solve) of a plan."""
    fp64 = precision == "fp64"
    if precision == "fp32_mfma":
        return False, False, False
    tiles = 16 <= n <= 2048
    lap = tiles if dims == 2 else 16 <= n <= (512 if fp64 else 1024) and not (fp64 and n == 256 and p <= 2)
    if dims == 2 and n >= 4096:
        lap = not fp64 and _pair(n, p, b)
    solve = tiles or (dims == 2 and (n == 4096 or (n == 8192 and not fp64)))
    return tiles, lap, solve


def _stages(pl, fn):
    pl.timing_reset()
    pl.timing(True)
    fn()
    pl.timing(False)
    torch.cuda.synchronize()
    st = pl.timing_read()
    pl.timing_reset()
    return st


@pytest.mark.parametrize("dims,n,p,b,batch,precision", PLANS)
def test_path_and_stage_record(dims, n, p, b, batch, precision):
    from stencilfft_amd import Plan
    print(f"[gpu] path {precision} {dims}D N={n} P={p} B={b} batch {batch}", flush=True)
    sys.stdout.flush()
    big = n ** dims * batch > 1 << 27  # the flags alone
    pl = Plan(dims, n, p, b, precision=precision, batch=batch, caller_scratch=big)
    tiles, lap, solve = _expected(dims, n, p, b, precision)
    assert (pl.tiled, pl.fused_laplace, pl.fused_solve) == (tiles, lap, solve)
    assert pl.fast == _pair(n, p, b)
    if big:
        return
    x = torch.zeros(pl.numel(), dtype=pl.complex_dtype, device="cuda")
    for fn in (pl.forward, pl.inverse):
        count, ms = _stages(pl, lambda: fn(x)).get("repack")
        assert count == dims - 1 and (ms == 0) == tiles
    st = _stages(pl, lambda: pl.laplace_forward(x))
    assert ("line_laplace" in st or st["laplace"] == (1, 0.0)) == lap, st
    st = _stages(pl, lambda: pl.spectral_solve(x, "heat", 1e-3, 1e-2))
    assert st["spectral"][0] == 1 and (st["spectral"][1] == 0) == solve, st
