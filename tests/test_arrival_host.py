"""CPU check of the last-workgroup test of the wide statistics (csrc/hip/arrival.hpp): the word that
hands the arrival number to the other waves is not used again before all of them have read it."""
import os
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.timeout(120)
def test_every_wave_reads_the_arrival_number():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "arrival_check")
        subprocess.run(["g++", "-std=c++17", "-O2", "-pthread", "-o", exe, os.path.join(HERE, "cpp", "arrival_check.cpp")],
                       check=True, timeout=100)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("OK"), r.stdout
