"""The lockstep reductions against host sums, and the iterate-only switch of the
Krylov solvers (tests/cpp/test_lockstep.hip, built with the library)."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
BIN = os.path.join(ROOT, "grid-mg-bench_amd", "bin", "test_lockstep")


def test_lockstep_reductions_and_iterates(gpu):
    assert os.path.exists(BIN), "build the package first (make -C grid-mg-bench_amd)"
    r = subprocess.run([BIN], capture_output=True, text=True, timeout=240)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert "ALL PASSED" in r.stdout
