"""GPU parity of the batched pentadiagonal ring kernels at the sizes where they
can go wrong: rows around whole chunks of 8 (and the last rows that do not
take the interior form), systems around whole blocks of 64, odd batches and
unaligned arrays (4-byte loads), and operands that leave the short division's
range.  The bar is bit equality with the CPU oracle."""
import numpy as np
import pytest

import oracle
from custen_amd import api
from tests.helpers import bits_equal, mismatches
from tests.test_oracle import _pent_systems

pytestmark = pytest.mark.gpu


def run(gpu, host, m, batch, shift=0):
    """Factor and solve on the device; shift: arrays start that many doubles
    past an aligned address."""
    dev = []
    for a in host:
        t = gpu.zeros(m * batch + shift, dtype=gpu.float64, device="cuda")[shift:]
        t.copy_(gpu.from_numpy(np.ascontiguousarray(a).ravel()))
        dev.append(t)
    api.custenPentFactorBatch(*dev[:5], m, batch)
    api.custenPentSolveBatch(*dev[:6], m, batch)
    gpu.cuda.synchronize()
    return [t.cpu().numpy().reshape(m, batch) for t in dev]


def check(got, host):
    fac = oracle.pent_factor_batch(*host[:5], nthreads=8)
    x = oracle.pent_solve_batch(*fac, host[5], nthreads=8)
    for name, g, ref in zip(("ds", "dl", "d", "du", "dw", "x"), got, list(fac) + [x]):
        assert bits_equal(g, ref), (name, mismatches(g, ref))


@pytest.mark.parametrize("m", [4, 5, 9, 10, 11, 12, 13, 18, 19, 20, 21, 26, 58, 59, 60, 67, 131])
@pytest.mark.parametrize("batch", [1, 2, 63, 64, 65, 130])
def test_row_and_block_remainders(gpu, m, batch):
    print(f"pent ring m={m} batch={batch}", flush=True)
    host = _pent_systems(m, batch, 40 * m + batch)
    check(run(gpu, host, m, batch), host)


@pytest.mark.parametrize("m", [4, 9, 12, 13, 35, 98])
@pytest.mark.parametrize("batch", [9000, 9001, 9025])
def test_wide_blocks(gpu, m, batch):
    """Enough systems for 64 per workgroup."""
    print(f"pent ring m={m} batch={batch}", flush=True)
    host = _pent_systems(m, batch, 40 * m + batch)
    check(run(gpu, host, m, batch), host)


@pytest.mark.parametrize("m,batch", [(20, 128), (77, 66), (20, 9000)])
def test_unaligned_arrays(gpu, m, batch):
    print(f"pent ring unaligned m={m} batch={batch}", flush=True)
    host = _pent_systems(m, batch, 7 * m)
    check(run(gpu, host, m, batch, shift=1), host)


@pytest.mark.parametrize("kind", ["zero_rhs", "tridiagonal", "tiny", "huge", "small_pivots"])
def test_operands_outside_the_short_division(gpu, kind):
    """Zero and signed-zero quotients, tiny and huge values, pivots below the
    short division's range: those rows take IEEE division."""
    print(f"pent ring {kind}", flush=True)
    m, batch = 45, 96
    host = [a.copy() for a in _pent_systems(m, batch, 77)]
    ds, dl, d, du, dw, b = host
    some = np.arange(batch) % 3 == 0
    if kind == "zero_rhs":
        b[:, some] = 0.0
        b[:, some & (np.arange(batch) % 2 == 0)] = -0.0
        b[20, :] = 0.0
    elif kind == "tridiagonal":
        ds[:, some] = 0.0
        dw[:, some] = -0.0
    elif kind == "tiny":
        b[:, some] *= 1e-300
        du[:, some] *= 1e-305
    elif kind == "huge":
        b[:, some] *= 1e300
    else:
        for a in (ds, dl, d, du, dw):
            a[:, some] *= 1e-200
    check(run(gpu, host, m, batch), host)


def test_rows_never_read(gpu):
    """ds of rows 0 and 1 and dl of row 0 take no part, whatever they hold."""
    m, batch = 30, 70
    host = [a.copy() for a in _pent_systems(m, batch, 5)]
    host[0][:2] = np.nan
    host[1][0] = np.nan
    got = run(gpu, host, m, batch)
    host[0][:2] = 0.0
    host[1][0] = 0.0
    ref = [a.copy() for a in host]
    fac = oracle.pent_factor_batch(*ref[:5], nthreads=8)
    x = oracle.pent_solve_batch(*fac, ref[5], nthreads=8)
    for g, r in ((got[2], fac[2]), (got[3], fac[3]), (got[4], fac[4]), (got[5], x)):
        assert bits_equal(g, r), mismatches(g, r)
