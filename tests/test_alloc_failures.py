"""Failing device allocations in the one-launch solves
(tests/cpp/alloc_demo.cc)."""
import os
import subprocess

import pytest

from lehrfempp_amd import build as B


def test_alloc_driver_compiles(tmp_path):
    cmd = B.alloc_demo_cmd(str(tmp_path / "alloc"))
    cmd.insert(cmd.index("-Wextra") + 1, "-Werror")
    res = subprocess.run(cmd, capture_output=True, text=True)
    assert res.returncode == 0, res.stderr[-4000:]


@pytest.mark.gpu
def test_alloc_driver_runs_on_gpu():
    assert os.path.exists(B.ALLOC_BIN), "build the driver first (python -m lehrfempp_amd.build)"
    res = subprocess.run([B.ALLOC_BIN], capture_output=True, text=True, timeout=100)
    print(res.stdout)
    assert res.returncode == 0, res.stdout + res.stderr
    assert "OK" in res.stdout
