"""Runs tests/cpp/test_wave_queue.hip: the persistent launches' work queue hands
out every schedule position once, and a lane that does not ask keeps its own.
The binary is built by __graft_entry__.build()."""
import os
import subprocess

import pytest

pytestmark = pytest.mark.gpu

BIN = os.path.join(os.path.dirname(os.path.abspath(__file__)), "cpp", "test_wave_queue.bin")


def test_wave_queue(gpu):
    assert os.path.exists(BIN), "build it with `python -m bacon_amd.build`"
    r = subprocess.run([BIN], capture_output=True, text=True, timeout=60)
    print(r.stdout)
    assert r.returncode == 0, r.stdout + r.stderr
