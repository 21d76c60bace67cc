"""launch_gemm with batches and K splits, on each of its kernels (tests/cpp/gemm_check.hip, built with the library)."""

import os
import subprocess

import pytest

CHECK = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "gemm_check")


@pytest.mark.gpu
def test_batches_and_splits():
    assert os.path.exists(CHECK), f"{CHECK} is missing: build with __graft_entry__.build()"
    r = subprocess.run([CHECK], capture_output=True, text=True, timeout=100)
    print(r.stdout, r.stderr, flush=True)
    assert r.returncode == 0, r.stdout + r.stderr
