"""GPU parity of batched passes of several steps at the sizes where their strips
and bands can go wrong: widths around one and two strips (120 stored
columns, 112 in FP32), odd widths (pairs of columns that straddle the wrap),
heights around bands and around the least height, one-sided windows, grids a pass leaves
out, FP32, and every remainder of the steps after whole passes.  Both sides are
compared bit for bit with the CPU oracle: the current field and the one before
the last step."""
import numpy as np
import pytest

import oracle
from custen_amd import api, synth
from tests.helpers import mismatches

pytestmark = pytest.mark.gpu


def compare_with_single_steps(gpu, sizes, steps, H, L, V, T, f32):
    dt = gpu.float32 if f32 else gpu.float64
    w = gpu.from_numpy(synth.uniform(H * V, 17, -0.3, 0.3)).cuda()
    ins = [gpu.rand(ny, nx, dtype=dt, device="cuda") for nx, ny in sizes]
    sides = []
    for single in (True, False):
        x = [t.clone() for t in ins]
        y = [gpu.zeros_like(t) for t in ins]
        b = api.Batch(y, x, w, H, L, V, T, f32=f32)
        for _ in range(steps if single else 1):
            b.run(1 if single else steps)
        gpu.cuda.synchronize()
        sides.append(x + y)
        b.close()
    assert all(gpu.equal(p, q) for p, q in zip(*sides))


def run(gpu, sizes, steps, H, L, V, T, f32=False, runs=1):
    """The given grids beside one that takes the batch past the L2s, without
    which it would take single steps."""
    dt = np.float32 if f32 else np.float64
    w = synth.uniform(H * V, 17, -0.3, 0.3)
    host = [synth.field(nx, ny, 200 + nx + ny).astype(dt) for nx, ny in sizes]
    ins = [gpu.from_numpy(f.copy()).cuda() for f in host]
    large = gpu.ones(3200 if f32 else 1600, 2048, dtype=ins[0].dtype, device="cuda")
    ins.append(large)
    outs = [gpu.zeros_like(t) for t in ins]
    b = api.Batch(outs, ins, gpu.from_numpy(w).cuda(), H, L, V, T, f32=f32)
    for _ in range(runs):
        b.run(steps)
    gpu.cuda.synchronize()
    side = b.parity
    assert side == (steps * runs) & 1
    for k, f in enumerate(host):
        prev = f
        for _ in range(steps * runs):
            prev, f = f, oracle.apply(f, w, H, L, V, T, True, nthreads=4)
        cur_got, prev_got = (outs[k], ins[k]) if side else (ins[k], outs[k])
        assert mismatches(cur_got.cpu().numpy(), f) == 0, sizes[k]
        assert mismatches(prev_got.cpu().numpy(), prev) == 0, sizes[k]
    b.close()


@pytest.mark.parametrize("nx", [127, 128, 129, 132, 223, 224, 225, 239, 240, 241, 360, 371])
def test_widths(gpu, nx):
    print(f"batch steps nx={nx}", flush=True)
    run(gpu, [(nx, 37)], 4, 5, 2, 5, 2)
    run(gpu, [(nx, 40)], 7, 3, 1, 3, 1)
    run(gpu, [(nx, 21)], 4, 5, 2, 5, 2, f32=True)


@pytest.mark.parametrize("ny", [9, 15, 16, 17, 18, 19, 20, 31, 32, 33, 63, 64, 65, 66, 70, 130])
def test_heights(gpu, ny):
    print(f"batch steps ny={ny}", flush=True)
    run(gpu, [(131, ny)], 4, 5, 2, 5, 2)
    run(gpu, [(131, ny)], 5, 3, 1, 3, 1)


@pytest.mark.parametrize("steps", [1, 2, 3, 4, 5, 6, 7, 8, 10])
@pytest.mark.parametrize("f32", [False, True])
def test_steps_and_left_out_grids(gpu, steps, f32):
    """Grids a pass takes beside narrow and low ones, run twice so that the
    second run starts from either side."""
    print(f"batch steps={steps} f32={f32}", flush=True)
    run(gpu, [(256, 48), (60, 100), (300, 12), (129, 33)], steps, 5, 2, 5, 2, f32, runs=2)


@pytest.mark.parametrize("H,L,V,T", [(5, 0, 5, 0), (5, 4, 5, 4), (5, 1, 5, 3), (3, 0, 3, 2),
                                     (3, 2, 3, 0)])
@pytest.mark.parametrize("nx", [130, 131, 365])
def test_one_sided_windows(gpu, H, L, V, T, nx):
    print(f"batch steps window {H},{L},{V},{T} nx={nx}", flush=True)
    run(gpu, [(nx, 29)], 4, H, L, V, T)
    run(gpu, [(nx, 29)], 4, H, L, V, T, f32=True)


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("H", [3, 5])
def test_long_bands(gpu, H, f32):
    """Enough waves for the longest bands, beside grids on either side of the
    sizes a pass takes, and batches on either side of the L2s."""
    print(f"batch steps long bands H={H} f32={f32}", flush=True)
    rest = [(515, 333), (100, 200), (4097, 70)]
    for sizes in ([(2048, 1200)] * 20 + rest, [(1024, 1024)] * 2 + rest,
                  [(1024, 1024)] * 9 + rest):
        compare_with_single_steps(gpu, sizes, 7, H, H // 2, H, H // 2, f32)
