"""A plan's tables: those its passes read and no others."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu


def test_device_memory_of_a_plan():
    """2048^2 FP64 on a caller's scratch: W_N (32 KiB), the row and the tile
    passes' twiddles (36 KiB each) and the half-angle sines (16 KiB), 120 KiB in
    one allocation.  The specialised pass's tables in two precisions and an FP32
    W_N would add 68 KiB; 20 KiB are left for rounding up."""
    from stencilfft_amd import Plan
    print("[gpu] device memory of 256 plans", flush=True)
    Plan(2, 2048, 8, 4, precision="fp64", caller_scratch=True).close()
    torch.cuda.synchronize()
    before = torch.cuda.mem_get_info()[0]
    plans = [Plan(2, 2048, 8, 4, precision="fp64", caller_scratch=True) for _ in range(256)]
    used = before - torch.cuda.mem_get_info()[0]
    for p in plans:
        p.close()
    assert used <= 256 * 140 * 1024, used / 256
