"""The table atan2 of the Birkhoff sums (henon_map_cpp_amd/csrc/hm_angle.h) is as
accurate as the library's atan2 that it stands for. Its last sum rounds by at most half
a unit in the last place (1 in units of 2^-53 of the result); what goes into it is below
2^-6 and carries roundings of 2.5 x 2^-53 of that: at most 2.5/64 of a unit for results
of 1 and, where the result is as small as 1/64 itself, up to 2.5. The mean is that of
correct rounding within a few per cent."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "henon_map_cpp_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
def test_mean_error_is_the_librarys(tmp_path):
    exe = str(tmp_path / "angle_mean_check")
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-std=c++17", "-I", CSRC,
                    os.path.join(HERE, "angle_mean_check.cpp"), "-o", exe], check=True)
    mean, library, worst = map(float, subprocess.run([exe], check=True, capture_output=True,
                                                     text=True).stdout.split())
    assert mean <= 1.03 * library
    assert worst <= 3.5
