"""The pool of freed device blocks, built for the CPU over a device that is
only bookkeeping (tests/pool): which requests reuse a block, the bound on what
is kept, what a request the device cannot fill does, when all goes back, that
no thread waits for another's wait for the device, and what happens without
host memory."""
import os
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "graph500_amd", "csrc")


@pytest.fixture(scope="module")
def binary(tmp_path_factory):
    out = str(tmp_path_factory.mktemp("pool") / "pool_check")
    subprocess.check_call(["g++", "-std=c++17", "-O1", "-g", "-Wall", "-pthread", "-I" + os.path.join(HERE, "pool"),
                           "-I" + CSRC, os.path.join(HERE, "pool", "pool_check.cc"), "-x", "c++",
                           os.path.join(CSRC, "g5_pool.hip"), "-o", out])
    return out


@pytest.mark.parametrize("check", ["sizes", "bound", "refill", "contexts", "buffer", "threads", "host_memory"])
def test_pool(binary, check):
    r = subprocess.run([binary, check], capture_output=True, text=True, timeout=20)
    assert r.returncode == 0, r.stderr
