"""What a handle reports of the kernel that Compute runs: custenGetBandMode and
mem_shared, without a configuration, with the caller's, and after tuning."""
import pytest

from custen_amd import api
from tests.test_gpu_stencil import create_weights

pytestmark = pytest.mark.gpu


def walker(H, V, rpw=4, size=8):
    return ((8 // rpw + 1) * rpw + V - 1) * (128 + 2 * (H & ~1)) * size


def strip(H, V, rpw=8, size=8):
    return (4 * rpw + V - 1) * ((128 + H + 1) & ~1) * size


def report(h):
    return api.custenGetBandMode(h), h.mem_shared


@pytest.mark.parametrize("variant,nx,ny,H,V,expected", [
    ("2DXYp", 300, 200, 5, 5, (1, walker(5, 5))),
    ("2DXYnp", 301, 99, 3, 3, (1, walker(3, 3))),
    ("2DXp", 128, 4, 5, 1, (0, strip(5, 1, 4))),      # four rows: too low for V + 4
    ("2DXp", 128, 5, 5, 1, (1, walker(5, 1))),
    ("2DYnp", 500, 30, 1, 9, (1, walker(1, 9))),
    ("2DXYp", 127, 300, 5, 5, (0, strip(5, 5, 4))),   # narrower than a strip
    ("2DXYnp", 131, 300, 5, 5, (0, strip(5, 5, 4))),  # its written window is
    ("2DXYp", 3000, 300, 9, 9, (1, walker(9, 9))),    # too few rows to stream
    ("2DXYnp", 4096, 4096, 9, 9, (1, 8 * 144 * 8)),   # rows streamed
])
def test_default(gpu, variant, nx, ny, H, V, expected):
    u = gpu.zeros(ny, nx, dtype=gpu.float64, device="cuda")
    w = gpu.ones(H * V, dtype=gpu.float64, device="cuda")
    h = api.cuSten_t()
    create_weights(variant, h, 1, nx, ny, gpu.zeros_like(u), u, w, H, H // 2, V, V // 2)
    assert report(h) == expected
    assert api.custenGetTileConfig(h) == (0, 0, 0)
    api.custenSetTileConfig(h, 8, 2)
    rpw = 4 if H == 9 else 8  # the widest shapes have one height
    assert report(h) == (0, strip(H, V, rpw))
    api.custenSetBandConfig(h, 4, 2)
    assert report(h) == (1, walker(H, V) if expected[0] else expected[1])
    api.custenSetTileConfig(h, 0, 0)
    assert report(h) == expected
    getattr(api, f"cuStenDestroy{variant}")(h)


def test_tuned(gpu):
    n = 1024
    u = gpu.rand(n, n, dtype=gpu.float64, device="cuda")
    w = gpu.ones(9, dtype=gpu.float64, device="cuda")
    h = api.cuSten_t()
    create_weights("2DXYp", h, 1, n, n, gpu.zeros_like(u), u, w, 3, 1, 3, 1)
    api.cuStenCompute2DXYp(h, api.DEVICE)
    gpu.cuda.synchronize()
    rpw = api.custenGetTileConfig(h)[0]
    band = api.custenGetBandMode(h)
    assert h.mem_shared == (walker(3, 3, rpw) if band else strip(3, 3, rpw))
    api.cuStenDestroy2DXYp(h)


def test_point_functions(gpu):
    """The xy built-ins run on the stencil kernels, the others do not."""
    nx, ny = 300, 90
    u = gpu.zeros(ny, nx, dtype=gpu.float64, device="cuda")
    out = gpu.zeros_like(u)
    c = gpu.ones(9, dtype=gpu.float64, device="cuda")
    h = api.cuSten_t()
    f = api.custenGetBuiltinFunction("xy_cube_minus")
    api.cuStenCreate2DXYpFun(h, 0, 1, nx, ny, 32, 32, out, u, c, 3, 1, 1, 3, 1, 1, f)
    assert report(h) == (1, walker(3, 3))
    api.cuStenDestroy2DXYpFun(h)
    f = api.custenGetBuiltinFunction("x_central_difference")
    api.cuStenCreate2DXpFun(h, 0, 1, nx, ny, 32, 32, out, u, c, 3, 1, 1, 1, f)
    assert api.custenGetBandMode(h) == 0
    api.cuStenDestroy2DXpFun(h)


def test_fp32(gpu):
    u = gpu.zeros(90, 300, dtype=gpu.float32, device="cuda")
    w = gpu.ones(25, dtype=gpu.float64, device="cuda")
    h = api.cuSten_t()
    api.custenCreate2DF32(h, 0, 1, 300, 90, 2, 1, gpu.zeros_like(u), u, w, 5, 2, 2, 5, 2, 2)
    assert report(h) == (1, walker(5, 5, size=4))
    api.custenDestroy2DF32(h)
