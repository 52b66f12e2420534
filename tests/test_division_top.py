"""The CH column solve's divisions (custen_amd/csrc/ch_kernels.hip) for numerators
from 2^900 up, on the CPU: the kernel has no upper limit for them and tells by a
step's last value whether one of its quotients left the finite range."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_finite_quotients_are_correctly_rounded(tmp_path):
    exe = tmp_path / "division_top_check"
    subprocess.run(["g++", "-O2", "-ffp-contract=off", "-std=c++17",
                    os.path.join(HERE, "cpu", "division_top_check.cpp"), "-o", str(exe)], check=True)
    five, two, rows = (tuple(map(int, line.split())) for line in subprocess.run(
        [str(exe), "2000000", "5"], capture_output=True, text=True, check=True,
        timeout=120).stdout.splitlines())
    for tried, finite, wrong in (five, two):
        assert tried >= 2000000 and finite > tried // 4 and wrong == 0
    assert rows[0] > 5000 and rows[1] == 0
