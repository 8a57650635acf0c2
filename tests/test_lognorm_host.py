"""The table logarithm of the MEGNO sums (henon_map_cpp_amd/csrc/hm_lognorm.h),
built for the host with g++ and checked against long double. Its roundings in
units of 2^-53 max(|result|, 1/4): the last sum 1, the table entry and the inner
sum 1/2 each (both below 2^-3), the product e log10(2)/2 1/2, the series and r
below 0.1: at most 2.6, held to 3."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "henon_map_cpp_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_half_log10_against_long_double(tmp_path):
    exe = str(tmp_path / "lognorm_check")
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-std=c++17", "-I", CSRC,
                    os.path.join(HERE, "lognorm_check.cpp"), "-o", exe], check=True)
    worst, ok = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()
    assert float(worst) <= 3.0
    assert ok == "1"
