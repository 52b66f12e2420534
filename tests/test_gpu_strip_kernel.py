"""GPU parity of the strip kernel, which handles take only when they ask for it
(or by the autotuner's choice): every variant, several strips, none of them
interior (odd widths), ragged last strips and bands, store masks, the zeroed
right columns of x-np, FP32 and the point-function built-ins.  Bit equality with
the CPU oracle, unwritten points untouched."""
import zlib

import numpy as np
import pytest

import oracle
from custen_amd import api, synth
from tests.helpers import mismatches
from tests.test_gpu_stencil import SENTINEL, create_weights, dev, oracle_weights

pytestmark = pytest.mark.gpu

CONFIGS = [(4, 1), (8, 2), (8, 4)]

SHAPES = [("2DXYp", 5, 2, 5, 2), ("2DXYnp", 5, 2, 5, 2), ("2DXYp", 3, 1, 3, 1),
          ("2DXYnp", 3, 0, 3, 2), ("2DXp", 9, 4, 1, 0), ("2DXnp", 7, 3, 1, 0),
          ("2DXnp", 5, 0, 1, 0), ("2DYp", 1, 0, 9, 4), ("2DYnp", 1, 0, 7, 6),
          ("2DXYnp", 9, 4, 9, 4), ("2DXYp", 7, 3, 7, 3), ("2DXYp", 3, 1, 5, 2),
          ("2DXYnp", 5, 2, 3, 1), ("2DXp", 13, 6, 1, 0), ("2DYnp", 1, 0, 11, 5),
          ("2DXYp", 1, 0, 1, 0)]


@pytest.mark.parametrize("variant,H,L,V,T", SHAPES)
@pytest.mark.parametrize("config", CONFIGS)
@pytest.mark.parametrize("nx,ny", [(640, 150), (641, 70), (777, 45), (1000, 33), (1001, 130)])
def test_weights(gpu, variant, H, L, V, T, config, nx, ny):
    print(f"strip kernel {variant} {H}x{V} {nx}x{ny} {config}", flush=True)
    seed = zlib.crc32(repr((variant, nx, ny, H, L, V, T)).encode()) & 0xFFFF
    u = synth.field(nx, ny, seed)
    w = synth.uniform(H * V, seed + 1, -2.0, 2.0)
    init = np.full_like(u, SENTINEL)
    du, out, dw = dev(gpu, u), dev(gpu, init), dev(gpu, w)
    h = api.cuSten_t()
    create_weights(variant, h, 1, nx, ny, out, du, dw, H, L, V, T)
    api.custenSetTileConfig(h, *config)
    assert api.custenGetBandMode(h) == 0
    getattr(api, f"cuStenCompute{variant}")(h, api.DEVICE)
    gpu.cuda.synchronize()
    getattr(api, f"cuStenDestroy{variant}")(h)
    ref = oracle_weights(variant, u, w, H, L, V, T, init)
    assert mismatches(out.cpu().numpy(), ref) == 0


@pytest.mark.parametrize("dir_,H,V", [(0, 5, 1), (1, 1, 5), (2, 5, 5), (2, 3, 3), (2, 9, 9)])
@pytest.mark.parametrize("periodic", [False, True])
@pytest.mark.parametrize("nx,ny", [(640, 70), (777, 45)])
@pytest.mark.parametrize("config", CONFIGS)
def test_fp32(gpu, dir_, H, V, periodic, nx, ny, config):
    print(f"strip kernel FP32 {dir_} {H}x{V} {nx}x{ny} {periodic} {config}", flush=True)
    seed = 11 * nx + ny + H
    u = synth.field(nx, ny, seed).astype(np.float32)
    w = synth.uniform(H * V, seed + 1, -2.0, 2.0)
    init = np.full_like(u, SENTINEL)
    du, out, dw = dev(gpu, u), dev(gpu, init), dev(gpu, w)
    h = api.cuSten_t()
    L, T = H // 2, V // 2
    api.custenCreate2DF32(h, 0, 1, nx, ny, dir_, int(periodic), out, du, dw, H, L, L, V, T, T)
    api.custenSetTileConfig(h, *config)
    api.custenCompute2DF32(h, api.DEVICE)
    gpu.cuda.synchronize()
    api.custenDestroy2DF32(h)
    ref = oracle.apply(u, w.astype(np.float32), H, L, V, T, periodic, out=init.copy(),
                       zero_right_edge=dir_ == 0 and not periodic)
    assert mismatches(out.cpu().numpy(), ref) == 0


@pytest.mark.parametrize("variant", ["2DXYpFun", "2DXYnpFun"])
@pytest.mark.parametrize("name", ["xy_weighted_sum", "xy_cube_minus"])
@pytest.mark.parametrize("nx,ny", [(640, 70), (777, 45)])
def test_point_functions(gpu, variant, name, nx, ny):
    print(f"strip kernel {variant} {name} {nx}x{ny}", flush=True)
    u = synth.field(nx, ny, nx)
    c = synth.uniform(9, 5, -1.0, 1.0)
    init = np.full_like(u, SENTINEL)
    du, out, dc = dev(gpu, u), dev(gpu, init), dev(gpu, c)
    f = api.custenGetBuiltinFunction(name)
    h = api.cuSten_t()
    getattr(api, f"cuStenCreate{variant}")(h, 0, 1, nx, ny, 32, 32, out, du, dc, 3, 1, 1, 3, 1, 1,
                                           f)
    api.custenSetTileConfig(h, 8, 2)
    getattr(api, f"cuStenCompute{variant}")(h, api.DEVICE)
    gpu.cuda.synchronize()
    getattr(api, f"cuStenDestroy{variant}")(h)
    v = ((u * u) * u) - u if name == "xy_cube_minus" else u
    ref = oracle.apply(v, c, 3, 1, 3, 1, variant == "2DXYpFun", out=init.copy())
    assert mismatches(out.cpu().numpy(), ref) == 0
