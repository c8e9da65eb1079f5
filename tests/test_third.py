"""Division by three in the mean flow and the turbulent energy (host side)."""
import os
import shutil
import subprocess

import pytest


def test_third_is_the_quotient(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe = tmp_path / "third_check"
    src = os.path.join(os.path.dirname(__file__), "third_check.cpp")
    subprocess.run([hipcc, "-std=c++17", "-O1", "-ffp-contract=off", "--offload-host-only", "-x", "hip", src,
                    "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout
