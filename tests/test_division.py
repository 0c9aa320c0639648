"""The division of the index maps (Div) on the host, compiled from the kernels' header."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_division_is_exact(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("no hipcc")
    exe = str(tmp_path / "division")
    subprocess.run([hipcc, "--offload-host-only", "-std=c++17", "-O2", "-w",
                    "-I", os.path.join(ROOT, "lettuce_amd", "csrc"),
                    os.path.join(ROOT, "tests", "cpp", "division.hip"), "-o", exe], check=True, timeout=300)
    out = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout
