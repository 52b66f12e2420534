"""Infinities and NaN in batched passes of several steps: beside the columns that
a strip computes and does not store, in the rows that bands repeat, and at the
wraps.  They spread by the stencil's extents and no further: values and places
are those of the CPU oracle's single steps."""
import numpy as np
import pytest

import oracle
from custen_amd import api, synth

pytestmark = pytest.mark.gpu


def same(got, ref):
    return np.array_equal(got, ref, equal_nan=True)


@pytest.mark.parametrize("f32", [False, True])
@pytest.mark.parametrize("H,L,V,T", [(5, 2, 5, 2), (3, 1, 3, 1), (5, 0, 5, 4), (3, 2, 3, 0)])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan])
@pytest.mark.parametrize("nx,ny", [(365, 150), (256, 40), (131, 17)])
def test_spread(gpu, f32, H, L, V, T, value, nx, ny):
    print(f"batch steps {value} f32={f32} {H}x{V} L={L} T={T} {nx}x{ny}", flush=True)
    dt = np.float32 if f32 else np.float64
    f = synth.field(nx, ny, 5).astype(dt)
    for x, y in ((0, 0), (nx - 1, ny // 2), (111, 3), (119, ny - 1), (120, 9), (127, 16),
                 (nx - 9, ny - 5), (nx // 2, 64)):
        if y < ny:
            f[y, x] = value
    w = synth.uniform(H * V, 17, -0.3, 0.3)
    ins = [gpu.from_numpy(f.copy()).cuda(),
           gpu.ones(3200 if f32 else 1600, 2048, dtype=gpu.float32 if f32 else gpu.float64,
                    device="cuda")]
    outs = [gpu.zeros_like(t) for t in ins]
    b = api.Batch(outs, ins, gpu.from_numpy(w).cuda(), H, L, V, T, f32=f32)
    b.run(4)  # one pass of three steps and a single one
    gpu.cuda.synchronize()
    assert b.parity == 0
    prev = f
    for _ in range(4):
        prev, f = f, oracle.apply(f, w, H, L, V, T, True, nthreads=4)
    assert same(ins[0].cpu().numpy(), f) and same(outs[0].cpu().numpy(), prev)
    assert np.isfinite(prev).any()
    b.close()
