"""GPU parity of the column solve where its sweeps begin, end and change over:
every number of rows left after the whole steps, factors that settle at every
step of the first ones or not at all, and fields with zeros, subnormal, huge and
not finite values, which leave the short divisions' range.  Bits are compared
with the CPU oracle (NaN only as NaN)."""
import numpy as np
import pytest

import oracle
from custen_amd import api, synth

pytestmark = pytest.mark.gpu


def check(n, c0, steps, **kw):
    s = api.CHSolver(api.ch_params(n, **kw), c0)
    s.run(steps)
    got = s.field()
    s.close()
    ref = oracle.CH(n, **kw)
    rc, rco = c0.ravel().copy(), c0.ravel().copy()
    with np.errstate(all="ignore"):
        ref.step(rc, rco, steps=steps)
    for g, r in zip(got, (rc, rco)):
        g, r = g.ravel(), r
        nan = np.isnan(r)
        assert np.array_equal(np.isnan(g), nan)
        assert np.array_equal(g.view(np.int64)[~nan], r.view(np.int64)[~nan])


def field(n, seed):
    return synth.uniform(n * n, seed, -0.1, 0.1).reshape(n, n)


@pytest.mark.parametrize("n", list(range(8, 56)) + list(range(124, 142)) + [277, 301])
def test_rows_left(gpu, n):
    print(f"ch column solve n={n}", flush=True)
    check(n, field(n, n), 3)
    check(n, field(n, n), 2, gamma=1e-4)


@pytest.mark.parametrize("n", [70, 98, 131, 200])
@pytest.mark.parametrize("gamma", [0.0, 1e-7, 1e-6, 1e-5, 3e-5, 1e-4, 3e-4, 1e-3, 3e-3, 1e-2, 0.1])
def test_change_over(gpu, n, gamma):
    print(f"ch column solve n={n} gamma={gamma}", flush=True)
    check(n, field(n, 3), 2, gamma=gamma)


@pytest.mark.parametrize("n", [64, 131])
@pytest.mark.parametrize("gamma", [0.01, 1e-4, 0.0])
def test_values(gpu, n, gamma):
    print(f"ch column solve values n={n} gamma={gamma}", flush=True)
    r = np.random.default_rng(5)
    check(n, np.zeros((n, n)), 2, gamma=gamma)
    for scale in (1e-310, 1e-300, 1e-272, 1e-160, 1e90, 1e100, 1e102, 1e103):
        check(n, field(n, 9) * scale, 1, gamma=gamma)
    c = field(n, 4)
    c[r.random((n, n)) < 0.6] = 0.0
    check(n, c, 2, gamma=gamma)
    for special in (np.inf, -np.inf, np.nan, 1e308, 1e154):
        c = field(n, 6)
        c[n // 3, n // 2] = special
        check(n, c, 1, gamma=gamma)
