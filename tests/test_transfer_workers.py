"""How many threads a field transfer takes (host side)."""
import os
import shutil
import subprocess

import pytest


def test_helpers_come_for_free_processors_only(tmp_path):
    cxx = shutil.which("g++") or shutil.which("c++")
    if not cxx:
        pytest.skip("no C++ compiler")
    exe = tmp_path / "transfer_workers_check"
    src = os.path.join(os.path.dirname(__file__), "transfer_workers_check.cpp")
    subprocess.run([cxx, "-std=c++17", "-O1", "-pthread", src, "-o", str(exe)], check=True, capture_output=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0 and r.stdout.strip().endswith("ok"), r.stdout
