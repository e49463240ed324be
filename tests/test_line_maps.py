"""The line passes' address maps against the layout algebra, on the CPU: every
valid (N, P, B) with N = 16 .. 256 in 2D and 16, 32 in 3D (tests/line_maps.cpp)."""
import os
import shutil
import subprocess

import pytest

from conftest import ROOT


def test_line_pass_address_maps(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("needs hipcc")
    exe = str(tmp_path / "line_maps")
    subprocess.run([hipcc, "--offload-arch=gfx950", "-O1", "-std=c++17", os.path.join(ROOT, "tests", "line_maps.cpp"),
                    "-o", exe], check=True, capture_output=True)
    res = subprocess.run([exe], capture_output=True, text=True)
    assert res.returncode == 0 and res.stdout.strip() == "103 shapes", res.stdout
