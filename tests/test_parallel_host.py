"""CPU check of the host loop over a call's tables (csrc/host/parallel.hpp): an exception in a worker
reaches the caller and too few threads slow the call down, where either used to end the process."""
import os
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.timeout(120)
def test_worker_exceptions_and_missing_threads():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "parallel_check")
        subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-o", exe, os.path.join(HERE, "cpp", "parallel_check.cpp")],
                       check=True, timeout=100)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("OK"), r.stdout
