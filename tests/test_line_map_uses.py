"""The converters' maps at the tile size that their kernel runs and the Laplacian
row passes' ends, against the layout algebra, on the CPU (tests/line_map_uses.cpp)."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT


def test_launched_address_maps(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("needs hipcc")
    exe = str(tmp_path / "line_map_uses")
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++17", os.path.join(ROOT, "tests", "line_map_uses.cpp"),
                    "-o", exe], check=True, capture_output=True)
    res = subprocess.run([exe], capture_output=True, text=True)
    assert res.returncode == 0 and res.stdout.strip() == "103 shapes", res.stdout
