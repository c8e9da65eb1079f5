"""Which wave of a tile moves which ghost chunk (host side)."""
import os
import shutil
import subprocess

import pytest


def test_every_chunk_is_moved_once(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    exe = tmp_path / "wave_plan_check"
    src = os.path.join(os.path.dirname(__file__), "wave_plan_check.cpp")
    subprocess.run([hipcc, "-std=c++17", "-O1", "--offload-host-only", "-x", "hip", src, "-o", str(exe)],
                   check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout
