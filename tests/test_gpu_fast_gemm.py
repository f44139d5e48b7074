"""Fast mode at many rows (fastg.hip, every dtype): x as three bf16 terms (q8_0, q4_0) or two f16 ones on the matrix cores.

Bounds. Against float64, the product of the dequantized weights: x is split exactly or to 2^-23 of each element, products
are exact, and what rounds is fp32 sums no longer than the exact mode's chains, so the relative error (2-norm) stays below
the exact mode's own on the same inputs (measured 0.3 to 0.7 of it); the test allows equality, largest row against largest
row. Per element the header's
bound, |a - b| / (1 + |b|) <= 1e-5 (q8_0, q4_0) / 1e-4 (q4_k, q6_k) of the oracle, at x1 and x1000."""
import numpy as np
import pytest

import oracle as O
from conftest import rel_err, same_bits
from tcb_amd import BF16, F16, F32, MODE_FAST, Q4, Q4K, Q6K, Q8, synth
from tcb_amd._lib import KNOB_FAST_GEMM

pytestmark = pytest.mark.gpu


@pytest.fixture(autouse=True)
def always_this_kernel(launch_shape):
    """The kernel's edges lie at sizes that a call would run on other kernels (K below 256 stays exact)."""
    launch_shape(KNOB_FAST_GEMM, 1)


TOL = {Q8: 1e-5, Q4: 1e-5, Q4K: 1e-4, Q6K: 1e-4}


def _call(backend, w, x, off, N, K, c0, row0, acc):
    M = x.shape[0]
    xb = backend.ctx.alloc(x.nbytes + 64)
    xb.upload(x, byte_offset=off)
    cb = backend.ctx.to_device(c0)
    (backend.Gemm if acc else backend.GemmSet)(M, N, K, (xb, off), w, cb, row0=row0, mode=MODE_FAST)
    got = cb.download(np.float32, M * N).reshape(M, N)
    xb.free()
    cb.free()
    return got


def _row_errors(y, x, deq):
    """Largest relative error (2-norm) of a row of y against float64; rows of zeros apart."""
    t = x.astype(np.float64) @ deq.astype(np.float64).T
    n = np.linalg.norm(t, axis=1)
    return float(np.max((np.linalg.norm(y - t, axis=1) / np.where(n > 0, n, 1))[n > 0]))


# q8_0 / q4_0: 32-, 64- and 128-row tiles, ragged rows and columns, ragged 64-element steps, K slices; K below 256 (exact)
SMALL = [(49, 33, 32, 0), (64, 257, 96, 3), (65, 256, 288, 0), (128, 300, 992, 1), (129, 255, 4096, 0), (50, 1030, 544, 2),
         (17, 14500, 4096, 0), (33, 8000, 4096, 0), (300, 20000, 288, 0), (129, 11487, 2400, 1)]
# k-quants: the smallest products that take this path
# (and 17 to 32 rows, where only the widest stores do)
LARGE = {Q4K: [(17, 700, 2304, 0), (32, 300, 4096, 3), (33, 513, 1024, 0), (129, 14336, 4096, 0), (460, 2051, 8192, 1), (64, 29000, 4096, 0), (2100, 14000, 256, 0)],
         Q6K: [(17, 700, 2304, 0), (32, 300, 4096, 3), (64, 513, 1024, 0), (130, 8000, 4096, 0), (260, 2051, 7680, 1), (32, 31000, 4096, 0), (1200, 13100, 256, 0)]}


@pytest.mark.parametrize("dt,M,N,K,row0", [(dt, *s) for dt in (Q8, Q4) for s in SMALL] +
                         [(dt, *s) for dt in (Q4K, Q6K) for s in LARGE[dt]])
def test_fast_gemm(backend, dt, M, N, K, row0):
    raw = synth.quant_weights(dt, row0 + N, K, seed=M + K, outliers=0.01)
    w = backend.FromQuantized(dt, raw, row0 + N, K)
    rows = np.ascontiguousarray(raw.reshape(row0 + N, -1)[row0:]).reshape(-1)
    x = synth.activations(M, K, seed=N)
    x[M // 2] = 0
    x[1] *= np.float32(1000)
    x[M - 1, K - 1] = np.nan
    c0 = synth.activations(M, N, seed=3)
    pick = sorted({0, 1, M // 2, M - 2, M - 1, min(M - 1, 31), min(M - 1, 32), min(M - 1, 63), min(M - 1, 64)})
    deq = O.dequant(dt, rows).reshape(N, K)
    for acc, off in ((False, 0), (True, 4)):
        got = _call(backend, w, x, off, N, K, c0, row0, acc)
        same_bits(got, _call(backend, w, x, off, N, K, c0, row0, acc))
        want = O.quant_gemm(dt, len(pick), N, K, x[pick], rows, c0[pick].reshape(-1) if acc else None).reshape(len(pick), N)
        for i, m in enumerate(pick):
            if m == M - 1:
                assert np.isnan(got[m]).all() and np.isnan(want[i]).all()
                continue
            scale = np.float32(1000 if m == 1 else 1)
            assert rel_err(got[m] / scale, want[i] / scale) <= TOL[dt], (m, acc)
            if m == M // 2:
                same_bits(got[m], c0[m] if acc else np.zeros(N, np.float32))
        if not acc:
            fin = [i for i, m in enumerate(pick) if m != M - 1]
            assert _row_errors(got[pick][fin], x[pick][fin], deq) <= _row_errors(want[fin], x[pick][fin], deq)
    w.release()


@pytest.mark.parametrize("dt", [Q8, Q4, Q4K, Q6K])
def test_fast_gemm_ranges(backend, dt):
    """One exponent per row: rows of huge, tiny and subnormal values, one huge element among tiny ones, Inf rows."""
    M, N, K = 300, (1024 if dt in (Q8, Q4) else 6600), 4096
    raw = synth.quant_weights(dt, N, K, seed=8, outliers=0.01)
    w = backend.FromQuantized(dt, raw, N, K)
    rng = np.random.default_rng(3)
    x = rng.standard_normal((M, K)).astype(np.float32)
    x[0] *= 1e30
    x[1] *= np.float32(1e-30)
    x[2] = x[2] * np.float32(1e-40)
    x[3, 5] = 1e4
    x[4, :256] *= np.float32(1e-20)
    x[5, 9] = np.inf
    x[6, 0] = -np.inf
    got = _call(backend, w, x, 0, N, K, np.zeros((M, N), np.float32), 0, False)
    want = O.quant_gemm(dt, 7, N, K, x[:7], raw).reshape(7, N)
    for m in range(7):
        assert np.array_equal(np.isnan(got[m]), np.isnan(want[m]))
        if m >= 5:
            assert np.array_equal(got[m][~np.isnan(want[m])], want[m][~np.isnan(want[m])])
            continue
        amax = float(np.max(np.abs(x[m])))
        if m == 2:  # results in the subnormal range: units of the last place
            assert float(np.max(np.abs(got[m].astype(np.float64) - want[m]))) <= K * 2.0 ** -149
        else:
            assert rel_err(got[m] / np.float32(amax), want[m] / np.float32(amax)) <= TOL[dt], m
    w.release()


@pytest.mark.parametrize("dt,M,I,K", [(Q8, 70, 300, 992), (Q4, 300, 130, 4096), (Q4K, 512, 1800, 4608), (Q6K, 300, 2000, 4096),
                                          (Q8, 33, 200, 512), (Q4, 70, 9000, 1024), (Q4K, 40, 300, 512), (Q6K, 20, 20000, 1280)])
def test_fast_gemm_swiglu(backend, dt, M, I, K):
    """The gate applied in the slice sum, or after the kernel where K is not sliced (K = 512, and more tiles than half the CUs),
    gives the bits of the product followed by the gate."""
    raw = synth.quant_weights(dt, 2 * I, K, seed=I, outliers=0.01)
    w = backend.FromQuantized(dt, raw, 2 * I, K)
    x = synth.activations(M, K, seed=K)
    gu = _call(backend, w, x, 0, 2 * I, K, np.zeros((M, 2 * I), np.float32), 0, False)
    xb, ob = backend.ctx.to_device(x), backend.ctx.alloc(M * I * 4)
    backend.GemmSwiGLU(M, K, xb, w, ob, mode=MODE_FAST)
    same_bits(ob.download(np.float32, M * I), O.swiglu(gu, M, I).reshape(-1))
    for b in (xb, ob):
        b.free()
    w.release()


def _outlier_case(dt, M, N, K, big):
    """x of order 1 with one element of `big` in every row; the weights at that element are zero, so no output depends on
    it. q4_k / q6_k, which keep 24 bits of a 256-element block's largest value: the whole block's are zero."""
    raw = synth.quant_weights(dt, N, K, seed=K + N, outliers=0.01)
    x = synth.activations(M, K, seed=M)
    k = K // 2 + 37
    rows = raw.reshape(N, -1)
    if dt == Q8:
        rows[:, k // 32 * 34 + 2 + k % 32] = 0
    elif dt == Q4:
        j = k // 32 * 18 + 2 + k % 16
        rows[:, j] = (rows[:, j] & 0xF0 | 8) if k % 32 < 16 else (rows[:, j] & 0x0F | 0x80)
    elif dt == Q4K:
        rows[:, k // 256 * 144 + 4:(k // 256 + 1) * 144] = 0  # scales, minimums and codes
    else:
        rows[:, k // 256 * 210:k // 256 * 210 + 192] = np.r_[np.zeros(128), np.full(64, 0xAA)].astype(np.uint8)  # codes 32
    assert not O.dequant(dt, raw).reshape(N, K)[:, k].any()
    x[:, k] = np.float32(big)
    return raw, x


@pytest.mark.parametrize("dt,M,N", [(Q8, 130, 1024), (Q4, 130, 1024), (Q4K, 300, 6400), (Q6K, 300, 4096)])
@pytest.mark.parametrize("big", [1e8, -1e20, 1e30, 3e38])
def test_fast_gemm_outlier(backend, dt, M, N, big):
    """The header's bound, |a - b| / (1 + |b|), unscaled, where one element is 1e8 to 3e38 times the others."""
    K = 4096
    raw, x = _outlier_case(dt, M, N, K, big)
    w = backend.FromQuantized(dt, raw, N, K)
    got = _call(backend, w, x, 0, N, K, np.zeros((M, N), np.float32), 0, False)
    pick = [0, 31, 32, M - 1]
    want = O.quant_gemm(dt, len(pick), N, K, x[pick], raw).reshape(len(pick), N)
    assert np.abs(want).max() > 0.1
    assert rel_err(got[pick], want) <= TOL[dt]
    w.release()


@pytest.mark.parametrize("dt", [Q8, Q4])
def test_fast_gemm_nonfinite_rows(backend, dt):
    """q8_0 / q4_0 take NaN and Inf as ordinary terms: every row non-finite in some way (NaNs whose payload is all in the low
    16 bits too), K in slices and not. A row's outputs are NaN or infinite where the oracle's are, its sign included."""
    for N, K in ((500, 4096), (300, 256)):
        M = 64
        raw = synth.quant_weights(dt, N, K, seed=5, outliers=0.01)
        w = backend.FromQuantized(dt, raw, N, K)
        x = synth.activations(M, K, seed=6)
        x.view(np.uint32)[np.arange(M), np.arange(M) * 3] = [(0x7F800001, 0xFFC00000, 0x7F800000, 0xFF800000)[m % 4] for m in range(M)]
        x[3::8, 200] = np.inf
        x[5] = np.nan
        got = _call(backend, w, x, 0, N, K, np.zeros((M, N), np.float32), 0, False)
        want = O.quant_gemm(dt, M, N, K, x, raw).reshape(M, N)
        assert np.array_equal(np.isnan(got), np.isnan(want))
        assert not np.isfinite(want).any() and np.array_equal(got[~np.isnan(want)], want[~np.isnan(want)])
        w.release()


def _with_scales(raw, d, dmin):
    r = raw.reshape(-1, 144).copy()
    for at, v in ((0, d), (2, dmin)):
        r[:, at:at + 2] = np.broadcast_to(np.asarray(v, np.float16), (len(r),)).copy().view(np.uint8).reshape(-1, 2)
    return r.reshape(-1)


@pytest.mark.parametrize("kind", ["random", "d = 0", "dmin = 0", "d < 0", "dmin < 0", "signs", "d << dmin", "dmin << d"])
@pytest.mark.parametrize("mean", [0, 3])
def test_fast_gemm_q4k_block_scales(backend, kind, mean):
    """q4_k blocks of random codes and 6-bit scales with block scales a quantizer would not write, for the kernel folds code and
    minimum terms through dmin m / d; x with a mean, so that the minimum term is large. Against float64 no further off
    than the exact mode (measured 0.3 to 0.7 of it)."""
    M, N, K = 260, 300, 4608
    nb = N * K // 256
    rng = np.random.default_rng(11)
    d, m = np.exp(rng.uniform(-9, -5, nb)), np.exp(rng.uniform(-9, -5, nb))
    sd, sm = rng.choice([-1, 1], nb), rng.choice([-1, 1], nb)
    d, m = {"random": (d, m), "d = 0": (0, m), "dmin = 0": (d, 0), "d < 0": (-d, m), "dmin < 0": (d, -m),
            "signs": (d * sd, m * sm), "d << dmin": (d / 1000, m), "dmin << d": (d, m / 1000)}[kind]
    raw = _with_scales(O.random_quant(Q4K, 7, nb), d, m)
    w = backend.FromQuantized(Q4K, raw, N, K)
    x = synth.activations(M, K, seed=1) + np.float32(mean)
    got = _call(backend, w, x, 0, N, K, np.zeros((M, N), np.float32), 0, False)
    pick = [0, 1, 31, 32, 127, 128, M - 1]
    want = O.quant_gemm(Q4K, len(pick), N, K, x[pick], raw).reshape(len(pick), N)
    deq = O.dequant(Q4K, raw).reshape(N, K)
    assert _row_errors(got[pick], x[pick], deq) <= _row_errors(want, x[pick], deq)
    w.release()


@pytest.mark.parametrize("xt,ct", [(BF16, BF16), (F16, F16), (BF16, F32), (F32, F16)])
@pytest.mark.parametrize("dt", [Q8, Q4, Q4K, Q6K])
def test_fast_gemm_typed(backend, dt, xt, ct):
    """16-bit x and c through the kernel: the bits of the fp32 call on the widened activations, rounded once."""
    M, N, K = 70, 300, 1024
    raw = synth.quant_weights(dt, N, K, seed=N, outliers=0.01)
    w = backend.FromQuantized(dt, raw, N, K)
    x, c0 = synth.activations(M, K, seed=K).reshape(-1), synth.activations(M, N, seed=N).reshape(-1)
    xa, ca = (x if xt == F32 else O.round16(xt, x)), (c0 if ct == F32 else O.round16(ct, c0))
    xw, cw = (x if xt == F32 else O.widen16(xt, xa)), (c0 if ct == F32 else O.widen16(ct, ca))
    for acc in (False, True):
        xb, cb = backend.ctx.to_device(xa), backend.ctx.to_device(ca)
        backend.GemmTyped(M, N, K, xb, xt, w, cb, ct, accumulate=acc, mode=MODE_FAST)
        got = cb.download(np.float32 if ct == F32 else np.uint16, M * N)
        want = _call(backend, w, xw.reshape(M, K), 0, N, K, cw.reshape(M, N), 0, acc).reshape(-1)
        if ct != F32:
            got, want = O.widen16(ct, got), O.widen16(ct, O.round16(ct, want))
        same_bits(got, want)
        for b in (xb, cb):
            b.free()
    w.release()
