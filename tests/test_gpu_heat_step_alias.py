"""heat_step with the input as output: refused before anything is launched, on
plans of both kinds (a two-stage plan's solve alone takes it)."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("two_stage", [False, True])
def test_input_as_output_is_refused(two_stage):
    from stencilfft_amd import Plan, ZmError
    from stencilfft_amd import _lib as L
    print(f"[gpu] heat step in place, two_stage={two_stage}", flush=True)
    pl = Plan(2, 256, 2, 8, precision="fp64", two_stage=two_stage)
    x = torch.full((pl.numel(),), 7.0 + 1.0j, dtype=torch.complex128, device="cuda")
    with pytest.raises(ZmError) as e:
        pl.heat_step(x, 1e-3, 1e-2, out=x)
    assert e.value.status == L.ZM_ERR_ALIAS
    torch.cuda.synchronize()
    assert bool((x == 7.0 + 1.0j).all())
    if two_stage:
        want = pl.spectral_solve(x, "heat", 1e-3, 1e-2)
        assert torch.equal(pl.spectral_solve(x, "heat", 1e-3, 1e-2, out=x), want)
