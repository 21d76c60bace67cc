"""The device block cache and the copy ring without a GPU: tests/cpp/buffers_check.cpp (built with the library) runs buffers.cpp over a
simulated device, one check per run."""

import os
import subprocess

import pytest

CHECK = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "buffers_check")


@pytest.mark.skipif(not os.path.exists(CHECK), reason="check not built")
@pytest.mark.parametrize("name", ["grow", "freed_block_in_pool", "other_contexts", "ring", "pinned"])
def test_buffers_on_a_simulated_device(name):
    r = subprocess.run([CHECK, name], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
