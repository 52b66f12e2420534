"""Which grids of a batch take several steps to a pass over memory (chooseSteps,
custen_amd/csrc/batch_rules.h), on the CPU."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def choose(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ not available")
    exe = tmp_path_factory.mktemp("rules") / "batch_rules_check"
    subprocess.run(["g++", "-O1", "-std=c++17", "-I/opt/rocm/include",
                    os.path.join(HERE, "cpu", "batch_rules_check.cpp"), "-o", str(exe)], check=True)

    def run(*grids, size=8, H=5, single=False):
        """(rows per band, stepped grids of each group); a group is (count, nx, ny)."""
        args = ["x".join(map(str, g)) for g in grids]
        out = subprocess.run([str(exe), str(size), str(H), str(int(single)), *args], check=True,
                             capture_output=True, text=True).stdout.split()
        return int(out[0]), [int(v) for v in out[1:]]

    return run


@pytest.mark.parametrize("size", [4, 8])
@pytest.mark.parametrize("H", [3, 5])
def test_a_batch_that_outgrows_the_caches(choose, size, H):
    grids = [(8, 2048, 2048), (3, 100, 500), (2, 500, 15)]
    assert choose(*grids, size=size, H=H)[1] == [8, 0, 0]
    assert choose((1, 1024, 1024), size=size, H=H)[1] == [0]


@pytest.mark.parametrize("size", [4, 8])
@pytest.mark.parametrize("H", [3, 5])
def test_a_configured_batch_takes_single_steps(choose, size, H):
    """The caller's tile configuration says how every step runs."""
    assert choose((8, 2048, 2048), size=size, H=H, single=True)[1] == [0]


@pytest.mark.parametrize("size", [4, 8])
def test_grids_whose_strips_double(choose, size):
    """A 5x5 grid of 128 columns takes two strips of a pass, as many points again
    as a single step computes: left out where such grids are most of the batch, not
    where they are few."""
    wide = [(80, 129, 300), (80, 256, 300)]
    assert choose((400, 128, 300), *wide, size=size, H=5)[1] == [0, 80, 80]
    assert choose((200, 128, 300), *wide, size=size, H=5)[1] == [200, 80, 80]
    assert choose((400, 128, 300), *wide, size=size, H=3)[1] == [400, 80, 80]
    assert choose((1000, 128, 300), size=size, H=5)[1] == [0]
    assert choose((1000, 128, 300), (1, 256, 300), size=size, H=5)[1] == [0, 0]


@pytest.mark.parametrize("size,H,grids,rows", [
    (4, 5, [(16, 1024, 1024)], 32), (4, 5, [(32, 1024, 1024)], 64), (4, 5, [(16, 2048, 2048)], 128),
    (8, 5, [(16, 1024, 1024)], 32), (8, 5, [(16, 2048, 2048)], 64), (8, 5, [(40, 2048, 2048)], 128),
    # tall grids beside low ones, whose waves are short
    (4, 5, [(4, 1024, 1024), (1000, 300, 20)], 32), (4, 3, [(7, 1024, 1024), (3000, 128, 20)], 32),
    (4, 5, [(7, 1024, 1024), (3500, 128, 16)], 16), (4, 3, [(1, 2048, 2048), (8000, 130, 20)], 32),
])
def test_rows_of_bands(choose, size, H, grids, rows):
    """Bands of the length that was measured as the fastest; in FP32 low grids' many
    short waves do not stand for tall grids' few long ones."""
    assert choose(*grids, size=size, H=H)[0] == rows
