"""The table atan2 of the Birkhoff sums (henon_map_cpp_amd/csrc/hm_angle.h), built
for the host with g++ and checked against long double. Its roundings in units of
2^-53 of the result: the octant's sum 1, the table entry and its sum with atan(u) at
most 2 together, u and its series at most 4 where the table entry is 0 (a result
that is u itself): held to 7."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "henon_map_cpp_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_angle_of_against_long_double(tmp_path):
    exe = str(tmp_path / "angle_check")
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-std=c++17", "-I", CSRC,
                    os.path.join(HERE, "angle_check.cpp"), "-o", exe], check=True)
    worst, ok = subprocess.run([exe], check=True, capture_output=True, text=True).stdout.split()
    assert float(worst) <= 7.0
    assert ok == "1"
