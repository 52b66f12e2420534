"""WENO tiles with a difference at the limit of the short flux form: a tile that
staged one evaluates all of its points operation by operation.  One such point at
the tiles' edges, corners and halos, just below, at and above the limits of both
square modes, in an otherwise ordinary field."""
import numpy as np
import pytest

from tests.test_gpu_weno_range import run, velocities

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("single,limit", [(True, 28), (False, 92)])
@pytest.mark.parametrize("rpw", [4, 8])
@pytest.mark.parametrize("x,y", [(0, 0), (61, 13), (63, 15), (64, 16), (66, 18), (67, 31), (129, 39),
                                 (100, 20)])
def test_one_wide_point(gpu, single, limit, rpw, x, y):
    print(f"weno wide point {x},{y} single={single} rpw={rpw}", flush=True)
    r = np.random.default_rng(x + 100 * y)
    ny, nx = 40, 130
    u, v = velocities(r, ny, nx)
    phi = r.integers(-8, 8, (ny, nx)) / 8.0
    around = 2.0 ** limit
    for value in (np.nextafter(around, 0), around, np.nextafter(around, np.inf), 16 * around, -around,
                  2.0 ** 100, np.inf, np.nan):
        f = phi.copy()
        f[y, x] = value
        run(gpu, f, u, v, 1.0, 1.0, single, rpw)
