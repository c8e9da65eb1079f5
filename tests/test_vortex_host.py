"""The initial vortex where its kernel cannot be launched (host side)."""
import os
import shutil
import subprocess

import pytest

import mrlbm


def test_tables_outlive_their_copy(tmp_path):
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(hipcc):
        pytest.skip("hipcc not available")
    mrlbm._lib.load()
    lib = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(mrlbm.__file__))), "libmrlbm.so")
    exe = tmp_path / "vortex_check"
    src = os.path.join(os.path.dirname(__file__), "vortex_check.cpp")
    subprocess.run([hipcc, "-std=c++17", "-O1", "--offload-host-only", "-x", "hip", src, "-x", "none", lib,
                    "-Wl,-rpath," + os.path.dirname(lib), "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout + r.stderr
