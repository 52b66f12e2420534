"""GPU parity of the band walker where its strips and bands do not line up with
the grid: widths around one and two strips (the last strip overlaps its
neighbour), odd widths and arrays that start one element past an aligned
address (element-aligned rows), heights around whole chunks, the zeroed right
columns of the non-periodic x variant, and the sizes below which the strip
kernel takes over.  Bit equality with the CPU oracle, unwritten points
untouched."""
import numpy as np
import pytest

import oracle
from custen_amd import api, synth
from tests.helpers import mismatches
from tests.test_gpu_stencil import SENTINEL, create_weights, oracle_weights

pytestmark = pytest.mark.gpu


def device(gpu, a, shift):
    t = gpu.zeros(a.size + shift, dtype=gpu.from_numpy(a).dtype, device="cuda")[shift:]
    t.copy_(gpu.from_numpy(np.ascontiguousarray(a)).view(-1))
    return t


def run(gpu, variant, nx, ny, H, L, V, T, config, shift=0):
    seed = 31 * nx + ny + 7 * H + V
    u = synth.field(nx, ny, seed)
    w = synth.uniform(H * V, seed + 1, -2.0, 2.0)
    init = np.full_like(u, SENTINEL)
    du, dout = device(gpu, u, shift), device(gpu, init, shift)
    dw = gpu.from_numpy(w).cuda()
    h = api.cuSten_t()
    create_weights(variant, h, 1, nx, ny, dout, du, dw, H, L, V, T)
    if config:
        api.custenSetBandConfig(h, *config)
    getattr(api, f"cuStenCompute{variant}")(h, api.DEVICE)
    gpu.cuda.synchronize()
    getattr(api, f"cuStenDestroy{variant}")(h)
    got = dout.cpu().numpy().reshape(ny, nx)
    assert mismatches(got, oracle_weights(variant, u, w, H, L, V, T, init)) == 0


SHAPES = [("2DXYp", 5, 2, 5, 2), ("2DXYnp", 5, 2, 5, 2), ("2DXYnp", 3, 2, 3, 0),
          ("2DXp", 7, 3, 1, 0), ("2DXnp", 7, 3, 1, 0), ("2DXnp", 9, 0, 1, 0),
          ("2DYp", 1, 0, 9, 4), ("2DYnp", 1, 0, 5, 1), ("2DXYnp", 9, 4, 9, 4),
          ("2DXYp", 7, 3, 7, 3)]


@pytest.mark.parametrize("variant,H,L,V,T", SHAPES)
@pytest.mark.parametrize("nx", [127, 128, 129, 131, 136, 137, 255, 257, 393])
def test_widths(gpu, variant, H, L, V, T, nx):
    print(f"band window {variant} {H}x{V} nx={nx}", flush=True)
    run(gpu, variant, nx, 45, H, L, V, T, (4, 2))
    run(gpu, variant, nx, 45, H, L, V, T, (4, 3), shift=1)


@pytest.mark.parametrize("variant,H,L,V,T", SHAPES)
@pytest.mark.parametrize("ny", [3, 4, 5, 8, 9, 11, 12, 13, 16, 17, 23, 24, 25, 33])
def test_heights(gpu, variant, H, L, V, T, ny):
    print(f"band window {variant} {H}x{V} ny={ny}", flush=True)
    for config in ((4, 1), (4, 4), (8, 2), None):
        run(gpu, variant, 259, ny, H, L, V, T, config)


@pytest.mark.parametrize("periodic", [True, False])
@pytest.mark.parametrize("nx,ny,H,V", [(129, 40, 5, 5), (261, 37, 3, 3), (255, 50, 7, 1),
                                       (387, 29, 1, 9), (200, 33, 9, 9)])
def test_f32(gpu, nx, ny, H, V, periodic):
    print(f"band window f32 {nx}x{ny} {H}x{V}", flush=True)
    u = synth.field(nx, ny, 5 * nx + ny).astype(np.float32)
    w = synth.uniform(H * V, 3, -1.0, 1.0)
    L, T = H // 2, V // 2
    dir_ = 2 if H > 1 and V > 1 else (0 if H > 1 else 1)
    init = np.full_like(u, np.float32(SENTINEL))
    for shift in (0, 1):
        du, dout = device(gpu, u, shift), device(gpu, init, shift)
        dw = gpu.from_numpy(w).cuda()
        h = api.cuSten_t()
        api.custenCreate2DF32(h, 0, 1, nx, ny, dir_, int(periodic), dout, du, dw, H, L, L, V, T, T)
        api.custenSetBandConfig(h, 4, 2)
        api.custenCompute2DF32(h, api.DEVICE)
        gpu.cuda.synchronize()
        api.custenDestroy2DF32(h)
        ref = oracle.apply(u, w, H, L, V, T, periodic,
                           zero_right_edge=not periodic and dir_ == 0, out=init.copy())
        assert mismatches(dout.cpu().numpy().reshape(ny, nx), ref) == 0


@pytest.mark.parametrize("nx,ny", [(129, 64), (257, 9), (128, 12), (641, 50), (64, 64)])
def test_batched_grids(gpu, nx, ny):
    """Grids walked whole beside grids the walker does not apply to."""
    sizes = [(nx, ny), (100, 33), (130, 31), (256, 5)]
    w = synth.uniform(25, 9, -0.2, 0.2)
    host = [synth.field(a, b, 100 + a + b) for a, b in sizes]
    ins = [gpu.from_numpy(f.copy()).cuda() for f in host]
    outs = [gpu.zeros_like(t) for t in ins]
    b = api.Batch(outs, ins, gpu.from_numpy(w).cuda())
    b.set_tile_config(4, 2, band=True)
    b.run(3)
    gpu.cuda.synchronize()
    for f, o in zip(host, outs):
        for _ in range(3):
            f = oracle.apply(f, w, 5, 2, 5, 2, True)
        assert mismatches(o.cpu().numpy(), f) == 0
    b.close()


ALIGNED = [("2DXYnp", 5, 2, 5, 2), ("2DXYnp", 3, 0, 3, 2), ("2DXYnp", 3, 2, 3, 1),
           ("2DXnp", 7, 3, 1, 0), ("2DXnp", 9, 0, 1, 0), ("2DXnp", 9, 8, 1, 0),
           ("2DXYnp", 9, 4, 9, 4), ("2DXYnp", 7, 0, 7, 6), ("2DYnp", 1, 0, 9, 4)]


@pytest.mark.parametrize("variant,H,L,V,T", ALIGNED)
@pytest.mark.parametrize("nx", [128, 144, 160, 240, 256, 272, 288, 384, 400, 416])
def test_aligned_rows(gpu, variant, H, L, V, T, nx):
    """Rows of whole lines: strips at multiples of 128 columns, the first and the
    last of the window drawn in."""
    print(f"band window aligned {variant} {H}x{V} L={L} nx={nx}", flush=True)
    run(gpu, variant, nx, 45, H, L, V, T, (4, 2))
    run(gpu, variant, nx, 45, H, L, V, T, (4, 8))
    run(gpu, variant, nx, 45, H, L, V, T, (8, 1), shift=1)
