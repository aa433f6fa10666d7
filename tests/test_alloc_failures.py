"""Failing allocations and refused launches in the one-launch solves
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


@pytest.mark.gpu
def test_alloc_driver_runs_beside_a_process_that_has_solved():
    # cooperative launches of a second process can be refused as long as the
    # first one lives
    import numpy as np

    from lehrfempp_amd import capi
    n = 4096
    i = np.arange(n)
    with capi.Context(0) as ctx:
        A = capi.coo_to_csr(ctx, np.concatenate([i, i[:-1], i[1:]]),
                            np.concatenate([i, i[1:], i[:-1]]),
                            np.concatenate([np.full(n, 2.1), np.full(2 * n - 2, -1.0)]), n, n)
        b, x = capi.Vec(ctx, np.ones(n)), capi.Vec(ctx, n)
        assert capi.pcg(ctx, A, b, x).syncs == 1
        test_alloc_driver_runs_on_gpu()
        x.fill(0.0)
        assert capi.pcg(ctx, A, b, x).syncs == 1
        for h in (x, b, A):
            h.close()
