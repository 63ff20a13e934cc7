"""Workgroups of the Krylov sweeps over the library's range of rows, columns and
Krylov dimensions (tests/cpp/sweep_check.cpp, built with the library).  CPU only."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("exe", ["sweep_check", "sweep_check_san"])
def test_sweep_blocks(exe):
    path = os.path.join(ROOT, "tests", "cpp", exe)
    assert os.path.exists(path), f"tests/cpp/{exe} is missing: run __graft_entry__.build()"
    out = subprocess.run([path], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout + out.stderr
