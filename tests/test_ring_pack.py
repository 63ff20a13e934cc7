"""The ring solve replayed on the host from the arrays that the upload sends
(tests/cpp/ring_check.cpp, built with the library): a step's rows written in
either order, ahead of or after the other rows' reads, give plain substitution; a
ring that is too short does not.  CPU only."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("exe", ["ring_check", "ring_check_san"])
def test_ring_slots(exe):
    path = os.path.join(ROOT, "tests", "cpp", exe)
    assert os.path.exists(path), f"tests/cpp/{exe} is missing: run __graft_entry__.build()"
    env = dict(os.environ, ASAN_OPTIONS="detect_leaks=0", UBSAN_OPTIONS="print_stacktrace=1:halt_on_error=1")
    out = subprocess.run([path], capture_output=True, text=True, timeout=600, env=env)
    print(out.stdout, out.stderr[-3000:])
    assert out.returncode == 0, out.stdout + out.stderr[-3000:]
    assert "controls detected" in out.stdout and "MISMATCH" not in out.stdout.split("control")[0]
