"""Workgroups of the Krylov sweeps over the library's range of rows, columns and
Krylov dimensions (tests/cpp/sweep_check.cpp, built with the library).  CPU only."""
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_sweep_blocks():
    path = os.path.join(ROOT, "tests", "cpp", "sweep_check")
    assert os.path.exists(path), "tests/cpp/sweep_check is missing: run __graft_entry__.build()"
    out = subprocess.run([path], capture_output=True, text=True, timeout=60)
    assert out.returncode == 0, out.stdout
