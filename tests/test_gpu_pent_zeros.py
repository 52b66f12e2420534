"""Batched factorisations whose quotients are exactly zero, in every row or in some,
of either sign and by pivots of either sign, beside quotients too small for the
short division: bit equality with the CPU oracle, signs of zeros included."""
import numpy as np
import pytest

from tests.test_gpu_pent_ring import check, run
from tests.test_oracle import _pent_systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("zero", [0.0, -0.0])
@pytest.mark.parametrize("sign", [1.0, -1.0])
@pytest.mark.parametrize("which", ["dw", "du", "du dw", "ds dw", "ds dl du dw", "some rows"])
@pytest.mark.parametrize("m,batch", [(45, 96), (67, 65), (30, 4099)])
def test_zero_quotients(gpu, which, sign, zero, m, batch):
    print(f"pent zeros {which} {sign} {zero} m={m} batch={batch}", flush=True)
    host = [a * sign for a in _pent_systems(m, batch, 3 * m)]
    named = dict(zip(("ds", "dl", "d", "du", "dw", "b"), host))
    if which == "some rows":
        named["dw"][::3] = zero
        named["du"][1::5] = zero
        named["dl"][1::5] = -zero
    else:
        for a in which.split():
            named[a][:] = zero
    check(run(gpu, host, m, batch), host)


@pytest.mark.parametrize("value", [5e-324, -5e-324, 1e-308, 2.0 ** -401, 2.0 ** -399])
def test_tiny_beside_zero(gpu, value):
    """One tiny entry in a chunk of zero quotients."""
    print(f"pent tiny beside zero {value}", flush=True)
    m, batch = 45, 70
    host = [a.copy() for a in _pent_systems(m, batch, 9)]
    host[4][:] = 0.0
    host[4][np.arange(m) % 7 == 3, ::2] = value
    host[3][:, ::3] = 0.0
    host[0][:, ::3] = 0.0
    check(run(gpu, host, m, batch), host)
