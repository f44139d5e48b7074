"""Exact products of more than 16 activation rows: passes of 16 or 32 rows, walked by one workgroup or dealt over
several, chunks whole or in slices. Bit-identical to the oracle whichever plan the sizes take (bit equality, so there is
no tolerance to choose)."""
import numpy as np
import pytest

import oracle as O
from conftest import same_bits
from tcb_amd import Q4, Q4K, Q6K, Q8, synth

pytestmark = pytest.mark.gpu

# (M, N, K): one row into the second tile, whole tiles of 16 and 32, a short last pass of each kind; one row block and a
# ragged one, many; K of one chunk, an odd number, more chunks than a workgroup's waves, a short last chunk (32-element
# formats)
SIZES = [(17, 64, 256), (32, 70, 1280), (33, 130, 2304), (48, 200, 4096), (77, 1000, 1024), (130, 96, 2560),
         (64, 10300, 512), (200, 4100, 256)]


@pytest.mark.parametrize("dt", [Q8, Q4, Q4K, Q6K])
@pytest.mark.parametrize("M,N,K", SIZES)
def test_rows_plan_bits(backend, dt, M, N, K):
    if dt in (Q8, Q4) and K > 256:
        K += 96
    raw = synth.quant_weights(dt, N, K, seed=N + K + M, outliers=0.01)
    w = backend.FromQuantized(dt, raw, N, K)
    x, c0 = synth.activations(M, K, seed=K + M), synth.activations(M, N, seed=N + 5).reshape(-1)
    # the last row's NaN and infinity stay in its own outputs
    x[M - 1, 3], x[M - 1, K - 1] = np.nan, np.inf
    xb, cb = backend.ctx.to_device(x), backend.ctx.to_device(c0)
    backend.Gemm(M, N, K, xb, w, cb)
    got = cb.download(np.float32, M * N).reshape(M, N)
    # the oracle on the rows where passes and tiles begin and end, and on the last
    rows = sorted({r for r in (0, 15, 16, 31, 32, 47, 48, 63, 64, 95, 96, 127, 128, M - 2, M - 1) if 0 <= r < M})
    want = O.quant_gemm(dt, len(rows), N, K, np.ascontiguousarray(x[rows]), raw,
                        np.ascontiguousarray(c0.reshape(M, N)[rows]).reshape(-1)).reshape(len(rows), N)
    same_bits(got[rows[:-1]], want[:-1])
    assert np.array_equal(np.isnan(got[M - 1]), np.isnan(want[-1]))
    assert np.isfinite(got[:M - 1]).all()
    for b in (xb, cb):
        b.free()
    w.release()
