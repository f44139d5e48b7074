"""Act-quant with a row's blocks dealt over the waves of a workgroup (actqw.hip) against the oracle, bit for bit: both sides
of every line of its dispatch (1, 16, 32 rows; 64- and 96-row tiles; four- and eight-wave workgroups, two column tiles),
row and column remainders, block counts around a round of 4 and 8, row slices, both accumulate modes, NaN / Inf rows."""
import numpy as np
import pytest

import oracle as O
from conftest import rel_err, same_bits
from tcb_amd import MODE_FAST, Q4K, Q6K

pytestmark = pytest.mark.gpu

SHAPES = [  # M, N, K, row0
    (1, 1, 256, 0), (1, 300, 2048, 3), (1, 77, 2304, 0), (1, 8195, 1280, 0), (2, 31, 4352, 1), (16, 100, 2304, 0),
    (15, 8193, 256, 0), (16, 8200, 2304, 2), (17, 33, 2304, 0), (32, 70, 256, 5), (31, 8250, 1024, 0),
    (33, 45, 2560, 0), (64, 130, 2304, 0), (96, 4100, 512, 1), (65, 4100, 2304, 0), (130, 33, 4352, 2),
    (40, 8300, 512, 0), (100, 8225, 768, 0),
    # two 96-row tiles, the second of two and of one 32-row tiles
    (130, 4090, 2304, 1), (97, 4090, 2560, 0)]


@pytest.mark.parametrize("dt", [Q4K, Q6K])
@pytest.mark.parametrize("M,N,K,row0", SHAPES)
def test_actq_blocks_bits(backend, dt, M, N, K, row0):
    rng = np.random.default_rng(M * 7 + N + K)
    raw = O.small_scale_quant(dt, M + N + K, (row0 + N) * K // 256)
    X = rng.standard_normal((M, K)).astype(np.float32)
    if M > 2:
        X[1] *= 1000
        X[2, :256] = 0
    if M > 6:
        X[M - 2, K - 1] = np.nan
        X[M // 2, 3] = np.inf
    c0 = rng.standard_normal(M * N).astype(np.float32)
    w = backend.FromQuantized(dt, raw, row0 + N, K)
    xb = backend.ctx.to_device(X)
    rows = np.ascontiguousarray(raw.reshape(row0 + N, -1)[row0:])
    for acc in (False, True):
        cb = backend.ctx.to_device(c0)
        backend.GemmActQuant(M, N, K, xb, w, cb, row0=row0, accumulate=acc)
        want = O.quant_gemm_act(dt, M, N, K, X, rows, c0 if acc else None)
        same_bits(cb.download(np.float32, M * N), want)
        if dt == Q4K:  # tolerance mode: the header's bound, rows scaled by 1000 against their size
            cb.upload(c0)
            backend.GemmActQuant(M, N, K, xb, w, cb, row0=row0, accumulate=acc, mode=MODE_FAST)
            got, ref = cb.download(np.float32, M * N).reshape(M, N), want.reshape(M, N)
            scale = np.where(np.arange(M) == 1, np.float32(1000 if M > 2 else 1), np.float32(1))[:, None]
            fin = np.isfinite(ref).all(axis=1)
            assert rel_err((got / scale)[fin], (ref / scale)[fin]) <= 1e-4
            assert np.array_equal(np.isnan(got[~fin]), np.isnan(ref[~fin]))
        cb.free()
    xb.free()
    w.release()


@pytest.mark.parametrize("dt", [Q4K, Q6K])
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_actq_one_bad_row(backend, dt, bad):
    """A single activation row holding NaN / Inf, quantized inside the kernel: the fp32 path's bits."""
    N, K = 50, 2304
    raw = O.small_scale_quant(dt, 5, N * K // 256)
    X = np.random.default_rng(3).standard_normal((1, K)).astype(np.float32)
    X[0, 2100] = bad
    w = backend.FromQuantized(dt, raw, N, K)
    xb, cb = backend.ctx.to_device(X), backend.ctx.alloc(N * 4)
    backend.GemmActQuant(1, N, K, xb, w, cb, accumulate=False)
    same_bits(cb.download(np.float32, N), O.quant_gemm_act(dt, 1, N, K, X, raw))
    for b in (xb, cb):
        b.free()
    w.release()


@pytest.mark.parametrize("dt", [Q4K, Q6K])
@pytest.mark.parametrize("N,K,at", [(4096, 2048, 0), (9000, 4096, 1024), (1500, 4096, 3000)])
def test_actq_token_over_its_input(backend, dt, N, K, at):
    """One row whose outputs lie over its activations (from element `at` on): x is read before any of them is written."""
    raw = O.small_scale_quant(dt, N, N * K // 256)
    w = backend.FromQuantized(dt, raw, N, K)
    x = np.random.default_rng(N).standard_normal(K).astype(np.float32)
    want = O.quant_gemm_act(dt, 1, N, K, x.reshape(1, K), raw)
    buf = backend.ctx.alloc((max(K, at + N) + 64) * 4)
    for _ in range(4):
        buf.upload(x)
        backend.GemmActQuant(1, N, K, buf, w, (buf, at * 4), accumulate=False)
        same_bits(buf.download(np.float32, N, byte_offset=at * 4), want)
    buf.free()
    w.release()
