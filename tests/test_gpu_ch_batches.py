"""Server lanes across their ways of enqueuing a batch of steps (launched one by
one at first, captured and replayed once batches repeat, a shorter last batch):
the fields have the bits of the single-simulation solver's."""
import numpy as np
import pytest

from custen_amd import api

pytestmark = pytest.mark.gpu


def field(n, seed):
    return np.random.default_rng(seed).uniform(-0.1, 0.1, (n, n))


@pytest.mark.parametrize("steps", [1, 8, 9, 10, 36, 45, 46, 54, 63, 64, 100, 200])
def test_steps(gpu, steps):
    print(f"ch batches steps={steps}", flush=True)
    srv = api.CHServer(budget_bytes=1 << 30, max_slots=8)
    sizes = [(48, steps), (48, max(1, steps - 7)), (65, steps), (65, 2 * steps)]
    ids = [srv.submit(api.ch_params(n), k, field(n, n + i)) for i, (n, k) in enumerate(sizes)]
    srv.run_until_idle()
    for i, (n, k) in enumerate(sizes):
        one = api.CHSolver(api.ch_params(n), field(n, n + i))
        one.run(k)
        assert np.array_equal(srv.result(ids[i]).view(np.int64), one.field()[0].view(np.int64)), (n, k)
    srv.close()


def test_late_request(gpu):
    """A request admitted to a lane whose batches are being replayed."""
    n = 64
    srv = api.CHServer(budget_bytes=1 << 30, max_slots=8)
    first = srv.submit(api.ch_params(n), 300, field(n, 1))
    for _ in range(30):
        srv.step()
    second = srv.submit(api.ch_params(n), 150, field(n, 2))
    srv.run_until_idle()
    for rid, k, seed in ((first, 300, 1), (second, 150, 2)):
        one = api.CHSolver(api.ch_params(n), field(n, seed))
        one.run(k)
        assert np.array_equal(srv.result(rid).view(np.int64), one.field()[0].view(np.int64))
    srv.close()
