"""The order in which a step's workgroups take the tiles (host side)."""
import os
import shutil
import subprocess

import pytest


def test_tile_order_is_a_permutation(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe = tmp_path / "xcd_order_check"
    src = os.path.join(os.path.dirname(__file__), "xcd_order_check.cpp")
    subprocess.run([hipcc, "-std=c++17", "-O1", "--offload-host-only", "-x", "hip", src, "-o", str(exe)],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout
