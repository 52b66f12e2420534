"""Rows that the strip kernel's tiles read on low periodic grids: the row map
over every tile height, window and grid height, on the CPU, and the kernel
itself against the oracle."""
import os
import shutil
import subprocess
import zlib

import numpy as np
import pytest

import oracle
from custen_amd import api, synth
from tests.helpers import mismatches
from tests.test_gpu_stencil import create_weights, dev

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.mark.skipif(shutil.which("g++") is None, reason="g++ not available")
def test_every_row_of_a_tile_is_in_the_grid(tmp_path):
    exe = tmp_path / "strip_rows_check"
    subprocess.run(["g++", "-O2", "-std=c++17", "-I/opt/rocm/include",
                    os.path.join(HERE, "cpu", "strip_rows_check.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout
    looked, outside, wrong, left = map(int, out.split())
    assert looked > 100000 and left > 100 and outside == 0 and wrong == 0


@pytest.mark.gpu
@pytest.mark.parametrize("variant,H,V", [("2DXp", 5, 1), ("2DYp", 1, 3), ("2DXYp", 5, 5),
                                         ("2DXYp", 3, 3), ("2DXYp", 9, 9)])
@pytest.mark.parametrize("rows", [0, 1, 3, 8])
@pytest.mark.parametrize("config", [None, (4, 1), (8, 4), (16, 1, 1)])
def test_low_periodic_grids(gpu, variant, H, V, rows, config):
    """Grids of the window's height and a little more, far lower than a tile."""
    nx, ny = 256, V + rows
    print(f"low grid {variant} {H}x{V} ny={ny} config={config}", flush=True)
    seed = zlib.crc32(repr((variant, H, V, rows)).encode()) & 0xFFFF
    u = synth.field(nx, ny, seed)
    w = synth.uniform(H * V, seed + 1, -1.0, 1.0)
    du, out, dw = dev(gpu, u), dev(gpu, np.zeros_like(u)), dev(gpu, w)
    h = api.cuSten_t()
    create_weights(variant, h, 1, nx, ny, out, du, dw, H, H // 2, V, V // 2)
    if config:
        api.custenSetTileConfig(h, *config)
    getattr(api, f"cuStenCompute{variant}")(h, api.DEVICE)
    gpu.cuda.synchronize()
    getattr(api, f"cuStenDestroy{variant}")(h)
    ref = oracle.apply(u, w, H, H // 2, V, V // 2, True)
    assert mismatches(out.cpu().numpy(), ref) == 0
