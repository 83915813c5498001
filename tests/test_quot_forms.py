"""The tail of the V-cycle forms quotients from kept reciprocals
(incrmt_amd/csrc/quot.hh). Within the range that the header states they must
equal the division bit for bit, and below and above it, where a remainder
underflows (the right-hand side of a single-precision cycle is an unscaled
residual), lie next to it; this compiles the product's header on the host and
checks both."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="no host compiler")
def test_quotients_are_the_division(tmp_path):
    exe = str(tmp_path / "quot_forms")
    subprocess.run(["g++", "-O2", "-std=c++17", "-ffp-contract=off", os.path.join(HERE, "quot_forms.cc"),
                    "-o", exe], check=True)
    r = subprocess.run([exe, "1000000"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    assert r.stdout.split() == ["0"] * 4
