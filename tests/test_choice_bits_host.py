"""CPU check of the merge loop with choice bits (the wave's table design) against std::pop_heap and
std::push_heap, lane by lane and with every heap access asserted in bounds."""
import os
import subprocess
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.timeout(300)
def test_choice_bits_match_std_library():
    with tempfile.TemporaryDirectory() as d:
        exe = os.path.join(d, "choice_check")
        subprocess.run(["g++", "-std=c++17", "-O2", "-o", exe, os.path.join(HERE, "cpp", "choice_check.cpp")],
                       check=True, timeout=240)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=240)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.startswith("OK"), r.stdout
