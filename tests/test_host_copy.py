"""The threaded host copy of served results (custen_amd/csrc/host_copy.h): sizes
around its splits, and no memory for some or all of its threads."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_copies_with_any_number_of_threads(tmp_path):
    exe = tmp_path / "host_copy_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-pthread",
                    os.path.join(HERE, "cpu", "host_copy_check.cpp"), "-o", str(exe)], check=True)
    copies, wrong, refused = map(int, subprocess.run([str(exe)], capture_output=True, text=True,
                                                     check=True, timeout=60).stdout.split())
    assert copies == 81 and wrong == 0 and refused > 10
