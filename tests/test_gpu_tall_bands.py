"""GPU parity of 1x13 as an untuned handle runs it, on both sides of the size from
which its bands are 12 rows: heights around the bands, odd widths, both boundary
modes and types.  The large grids are compared with the strip kernel, which has
its own parity tests; points that Compute does not write are untouched."""
import pytest

from custen_amd import api, synth
from tests.test_gpu_stencil import create_weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("periodic", [0, 1])
@pytest.mark.parametrize("nx,ny", [(2048, 2047), (2048, 2048), (2048, 2049), (1999, 2101),
                                   (2000, 2110), (2001, 2123), (131, 32100), (240000, 18)])
def test_default(gpu, monkeypatch, f32, periodic, nx, ny):
    print(f"tall bands {nx}x{ny} f32={f32} periodic={periodic}", flush=True)
    monkeypatch.setenv("CUSTEN_AUTOTUNE", "0")
    u = gpu.rand(ny, nx, dtype=gpu.float32 if f32 else gpu.float64, device="cuda")
    w = gpu.from_numpy(synth.uniform(13, 3, -1.0, 1.0)).cuda()
    variant = "2DYp" if periodic else "2DYnp"
    outs = []
    for config in (None, (4, 1)):
        out = gpu.full_like(u, 7.0)
        h = api.cuSten_t()
        if f32:
            api.custenCreate2DF32(h, 0, 1, nx, ny, 1, periodic, out, u, w, 1, 0, 0, 13, 6, 6)
        else:
            create_weights(variant, h, 1, nx, ny, out, u, w, 1, 0, 13, 6)
        if config:
            api.custenSetTileConfig(h, *config)
        assert api.custenGetBandMode(h) == (0 if config else 1)
        getattr(api, "custenCompute2DF32" if f32 else f"cuStenCompute{variant}")(h, api.DEVICE)
        gpu.cuda.synchronize()
        getattr(api, "custenDestroy2DF32" if f32 else f"cuStenDestroy{variant}")(h)
        outs.append(out)
    assert gpu.equal(*outs)
