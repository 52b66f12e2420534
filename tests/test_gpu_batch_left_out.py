"""Grids that batched passes of several steps leave out (narrow ones, low ones) take
their single steps with the tuned configuration, the band walker where it
applies.  The choice is given through a tuning file, in a child process, and the
results are compared bit for bit with configured single steps."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

CHILD = """
import sys
sys.path.insert(0, %r)
import torch
from custen_amd import api

# (ny, nx) beside one or two grids that take passes
REST = [(12, 4096), (15, 1000), (9, 128), (8, 300), (4, 200), (3, 500), (100, 60), (300, 128),
        (5, 7), (13, 131)]
for f32 in (False, True):
    for H in (3, 5):
        shapes = [(2048, 2200)] * (2 if f32 else 1) + REST
        dt = torch.float32 if f32 else torch.float64
        torch.manual_seed(H)
        start = [torch.rand(s, device='cuda', dtype=dt) for s in shapes]
        w = torch.rand(H * H, device='cuda', dtype=torch.float64) - 0.5
        sides = []
        for single in (False, True):
            a = [t.clone() for t in start]
            b = [torch.zeros_like(t) for t in a]
            batch = api.Batch(b, a, w, H, H // 2, H, H // 2, f32=f32)
            if single:
                batch.set_tile_config(4, 1)
            batch.run(5)
            batch.run(7)
            torch.cuda.synchronize()
            config = batch.tile_config()
            batch.close()
            sides.append(a + b)
            print('case', f32, H, single, *config, flush=True)
        print('differ', sum(not torch.equal(x, y) for x, y in zip(*sides)), flush=True)
"""


@pytest.mark.parametrize("config", ["4 2 2 1", "8 1 2 1", "8 4 2 0"])
def test_left_out_grids(gpu, tmp_path, config):
    from custen_amd import api  # noqa: F401  (the library is there)

    rest = 12 * 4096 + 15 * 1000 + 9 * 128 + 8 * 300 + 4 * 200 + 3 * 500 + 6000 + 300 * 128 + 35 + \
        13 * 131
    cache = tmp_path / "tune.txt"
    lines = []
    for f32 in (0, 1):
        n = 2 if f32 else 1
        for H in (3, 5):
            lines.append(f"1 {f32} {H} {H} 0 {(n * 2048 * 2200 + rest) >> 20} 4096 {n + 10} {config}")
    cache.write_text("\n".join(lines) + "\n")
    r = subprocess.run([sys.executable, "-c", CHILD % ROOT], capture_output=True, text=True,
                       env=dict(os.environ, CUSTEN_TUNE_CACHE=str(cache)), timeout=60)
    print(r.stdout, flush=True)
    assert r.returncode == 0, r.stderr[-2000:]
    assert r.stdout.count("differ 0") == 4
    rpw, chunks, _, band = config.split()
    for f32 in (False, True):
        for H in (3, 5):
            assert f"case {f32} {H} False {rpw} {chunks} {band}\n" in r.stdout
    assert cache.read_text().strip().splitlines() == lines  # nothing was tuned
