"""GPU parity of the WENO advection kernel where its short forms end: tiles and
their remainders, and fields whose differences are zero, subnormal, beyond the
range of the short divisions, near overflow or not finite, which a wave
evaluates again operation by operation."""
import numpy as np
import pytest

import oracle
from custen_amd import api

pytestmark = pytest.mark.gpu


def run(gpu, phi, u, v, dx, dy, single, rpw=0):
    ny, nx = phi.shape
    d = [gpu.from_numpy(t.copy()).cuda() for t in (phi, u, v)]
    out = gpu.full_like(d[0], 7.0)
    h = api.cuSten_t()
    api.cuStenCreate2DXYWENOADVp(h, 0, 1, nx, ny, 32, 32, dx, dy, d[1], d[2], out, d[0])
    api.custenSetWenoSquares(h, single)
    if rpw:
        api.custenSetTileConfig(h, rpw, 1)
    api.cuStenCompute2DXYWENOADVp(h, api.DEVICE)
    gpu.cuda.synchronize()
    api.cuStenDestroy2DXYWENOADVp(h)
    with np.errstate(all="ignore"):
        ref = oracle.weno(phi, u, v, dx, dy, single, nthreads=8)
    got = out.cpu().numpy()
    nan = np.isnan(ref)
    assert np.array_equal(np.isnan(got), nan)
    assert np.array_equal(got.view(np.int64)[~nan], ref.view(np.int64)[~nan])


def velocities(r, ny, nx):
    u, v = r.uniform(-1, 1, (2, ny, nx))
    u[r.random((ny, nx)) < 0.1] = 0.0
    return u, v


@pytest.mark.parametrize("nx", [1, 2, 5, 63, 64, 65, 130])
@pytest.mark.parametrize("ny", [1, 3, 15, 16, 17, 31, 32, 33, 65])
def test_tiles(gpu, nx, ny):
    print(f"weno tiles {nx}x{ny}", flush=True)
    r = np.random.default_rng(nx * 100 + ny)
    u, v = velocities(r, ny, nx)
    phi = r.uniform(-1, 1, (ny, nx))
    for rpw in (4, 8):
        run(gpu, phi, u, v, 0.1, 0.2, True, rpw)
        run(gpu, phi, u, v, 0.1, 0.2, False, rpw)


# scales of the differences: subnormal, tiny, around 1, around the limits of the
# short divisions (squares of 2^60 and 2^190), around the overflow of a square
# in single and in double precision, and around that of a difference itself
SCALES = [2.0 ** k for k in (-1074, -1060, -600, -500, -149, -80, -30, 0, 14, 28, 29, 30, 31, 32, 33,
                             60, 63, 64, 65, 93, 94, 95, 96, 97, 255, 256, 510, 511, 512, 1020,
                             1021, 1022, 1023)]


@pytest.mark.parametrize("single", [True, False])
@pytest.mark.parametrize("scale", SCALES)
def test_scales(gpu, scale, single):
    print(f"weno scale {scale} single={single}", flush=True)
    r = np.random.default_rng(7)
    ny, nx = 40, 200
    u, v = velocities(r, ny, nx)
    phi = r.uniform(-1, 1, (ny, nx)) * scale
    phi[:, 64:128] = scale * (r.random((ny, 64)) < 0.3)  # steps: many zero differences
    run(gpu, phi, u, v, 1.0, 1.0, single)
    # nearly equal differences of that size, of both signs
    ramp = np.cumsum(np.ones((ny, nx)), axis=1) % 5 - 2 + 1e-3 * r.uniform(-1, 1, (ny, nx))
    run(gpu, ramp * (scale / 4), u, v, 1.0, 1.0, single)
    run(gpu, phi / scale if scale > 1e-300 else phi, u, v, 1.0 / max(scale, 1e-300),
        3.0, single)


@pytest.mark.parametrize("single", [True, False])
def test_mixed_and_not_finite(gpu, single):
    print(f"weno mixed single={single}", flush=True)
    r = np.random.default_rng(11)
    ny, nx = 96, 300
    u, v = velocities(r, ny, nx)
    phi = r.uniform(-1, 1, (ny, nx)) * r.choice(SCALES, (ny, nx))
    run(gpu, phi, u, v, 1.0, 0.5, single)
    phi = r.uniform(-1, 1, (ny, nx))
    at = r.random((ny, nx))
    phi[at < 0.01] = np.inf
    phi[at > 0.99] = -np.inf
    phi[(at > 0.5) & (at < 0.505)] = np.nan
    u[5, :] = np.nan
    v[7, 3] = np.inf
    run(gpu, phi, u, v, 1.0, 0.5, single)
