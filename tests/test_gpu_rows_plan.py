"""Exact products of more than 16 activation rows: passes of 16 or 32 rows, walked by one workgroup or dealt over
several, chunks whole or in slices. Bit-identical to the oracle with the plan the sizes take and with each kind of plan
forced (bit equality, so there is no tolerance to choose)."""
import numpy as np
import pytest

import oracle as O
from conftest import same_bits
from tcb_amd import BF16, F16, F32, MODE_EXACT, Q4, Q4K, Q6K, Q8, synth
from tcb_amd._lib import KNOB_ROWS

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


@pytest.mark.parametrize("xt,ct", [(F16, F16), (BF16, BF16), (F32, F16), (BF16, F32)])
@pytest.mark.parametrize("dt,M,N,K,off", [(Q8, 2, 300, 4096, 0), (Q4K, 6, 130, 2048, 2), (Q6K, 13, 64, 512, 6),
                                          (Q4, 40, 200, 2560, 0), (Q4K, 33, 10300, 256, 0)])
def test_rows_typed_bits(backend, xt, ct, dt, M, N, K, off):
    """16-bit x widened as it is staged and 16-bit c rounded as it is written (by the product or by the sum of its
    slices), x off the kernel's alignment included: the bits of the fp32 call on the widened activations, rounded."""
    raw = synth.quant_weights(dt, N, K, seed=N + K, outliers=0.01)
    w = backend.FromQuantized(dt, raw, N, K)
    x, c0 = synth.activations(M, K, seed=K + M).reshape(-1), synth.activations(M, N, seed=N).reshape(-1)
    x[K + 1], c0[5] = np.nan, np.inf
    xa = x if xt == F32 else O.round16(xt, x)
    ca = c0 if ct == F32 else O.round16(ct, c0)
    xw, cw = x if xt == F32 else O.widen16(xt, xa), c0 if ct == F32 else O.widen16(ct, ca)
    off *= 2 if xt == F32 else 1
    xb = backend.ctx.alloc(xa.nbytes + 64)
    xb.upload(xa, byte_offset=off)
    cb, x32, c32 = backend.ctx.to_device(ca), backend.ctx.to_device(xw), backend.ctx.to_device(cw)
    backend.GemmTyped(M, N, K, (xb, off), xt, w, cb, ct, accumulate=True, mode=MODE_EXACT)
    backend.Gemm(M, N, K, x32, w, c32)
    got, want = cb.download(np.float32 if ct == F32 else np.uint16, M * N), c32.download(np.float32, M * N)
    if ct != F32:
        got, want = O.widen16(ct, got), O.widen16(ct, O.round16(ct, want))
    same_bits(got, want)
    for b in (xb, cb, x32, c32):
        b.free()
    w.release()


# chunks whole (one or two turns of a workgroup's eight waves, the second short) or in slices (several turns of four);
# passes of 16 and 32 rows, all walked by one workgroup, dealt one each, and several each
PLANS = [(1, 16, 1), (1, 16, 3), (1, 32, 1), (1, 32, 2), (1, 32, 99), (2, 16, 1), (2, 16, 2), (2, 32, 1), (2, 32, 2), (2, 32, 99)]


@pytest.mark.parametrize("dt", [Q8, Q4, Q4K, Q6K])
@pytest.mark.parametrize("plan", PLANS)
@pytest.mark.parametrize("M,N,K", [(97, 130, 2304), (49, 70, 4352), (41, 64, 1280)])  # last 32-row pass of 1, 17, 9 rows
def test_forced_plan_bits(backend, launch_shape, dt, plan, M, N, K):
    if dt in (Q8, Q4):
        K += 96  # a short last chunk
    raw = synth.quant_weights(dt, N, K, seed=N + K + M, outliers=0.01)
    w = backend.FromQuantized(dt, raw, N, K)
    x, c0 = synth.activations(M, K, seed=K + M), synth.activations(M, N, seed=N + 5).reshape(-1)
    want = O.quant_gemm(dt, M, N, K, x, raw, c0)
    h, hc = O.round16(BF16, x.reshape(-1)), O.round16(BF16, c0)
    want16 = O.round16(BF16, O.quant_gemm(dt, M, N, K, O.widen16(BF16, h).reshape(M, K), raw, O.widen16(BF16, hc)))
    xb, cb, hb, hcb = (backend.ctx.to_device(v) for v in (x, c0, h, hc))
    launch_shape(KNOB_ROWS, *plan)
    backend.Gemm(M, N, K, xb, w, cb)
    same_bits(cb.download(np.float32, M * N), want)
    backend.GemmTyped(M, N, K, hb, BF16, w, hcb, BF16, accumulate=True, mode=MODE_EXACT)
    same_bits(O.widen16(BF16, hcb.download(np.uint16, M * N)), O.widen16(BF16, want16))
    for b in (xb, cb, hb, hcb):
        b.free()
    w.release()


@pytest.mark.parametrize("dt", [Q8, Q4, Q4K, Q6K])
@pytest.mark.parametrize("M,N,K,at", [(3, 256, 256, 0), (20, 300, 512, 1000), (5, 70, 2304, 5000)])
def test_rows_typed_over_its_input(backend, dt, M, N, K, at):
    """c over x (from element `at` on): the call reads all of x, through its fp32 copy, before it writes c."""
    raw = synth.quant_weights(dt, N, K, seed=N + K, outliers=0.01)
    w = backend.FromQuantized(dt, raw, N, K)
    h = O.round16(BF16, synth.activations(M, K, seed=K).reshape(-1))
    want = O.widen16(BF16, O.round16(BF16, O.quant_gemm(dt, M, N, K, O.widen16(BF16, h).reshape(M, K), raw)))
    buf = backend.ctx.alloc((max(M * K, at + M * N) + 64) * 2)
    for _ in range(3):
        buf.upload(h)
        backend.GemmTyped(M, N, K, buf, BF16, w, (buf, 2 * at), BF16, accumulate=False, mode=MODE_EXACT)
        same_bits(O.widen16(BF16, buf.download(np.uint16, M * N, byte_offset=2 * at)), want)
    buf.free()
    w.release()
