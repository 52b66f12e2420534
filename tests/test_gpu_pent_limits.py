"""Batched pentadiagonal systems on both sides of the batch sizes at which the
kernels change (16 and 64 systems to a workgroup, ring and one-wave kernels), even
and odd: bit equality with the CPU oracle."""
import pytest

from tests.test_gpu_pent_ring import check, run
from tests.test_oracle import _pent_systems

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [4, 13, 35])
@pytest.mark.parametrize("batch", [4095, 4097, 8192, 8193, 16384, 16385, 16386, 32767, 32768, 32769, 32770])
def test_around_the_limits(gpu, m, batch):
    print(f"pent limits m={m} batch={batch}", flush=True)
    host = _pent_systems(m, batch, m + batch)
    check(run(gpu, host, m, batch), host)
