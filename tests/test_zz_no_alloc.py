"""The allocation-free act-quant entry point (trhip_gemm_q_actq_noalloc, static device scratch) through the C-ABI:
the same bits as trhip_gemm_q_actq on calls in a row, each smaller than the one before (so the scratch holds the last
call's contents; one q4_k call takes the tiled 128-row prefill kernel), in set and accumulate mode, with an unaligned
activation pointer and a NaN row, and sizes beyond the scratch refused before anything runs."""
import ctypes

import numpy as np
import pytest

import oracle as O
from conftest import same_bits
from tcb_amd import Q4, Q4K, Q6K, QuantBackend, _lib, synth

pytestmark = pytest.mark.gpu

CASES = {Q4K: [(512, 4096, 4096), (256, 24576, 1024), (40, 300, 2048)], Q4: [(96, 1024, 4096), (9, 130, 1024)],
         Q6K: [(64, 1024, 4096), (5, 77, 2048)]}


@pytest.mark.parametrize("dt", [Q4K, Q4, Q6K])
def test_noalloc_matches_actq(backend, dt):
    L = _lib.lib()
    h = backend.ctx.h
    for i, (M, N, K) in enumerate(CASES[dt]):
        print("noalloc case dt=%d M=%d N=%d K=%d" % (dt, M, N, K), flush=True)
        raw = synth.quant_weights(dt, N, K, seed=90 + i, outliers=0.01 if dt != Q4 else 0.0)
        w = backend.FromQuantized(dt, raw, N, K)
        X = synth.activations(M, K, seed=91 + i)
        X[M // 2, 7] = np.nan
        off = 4 * i  # the second call takes an x that is not 16-byte aligned (copied inside the scratch)
        xb = backend.ctx.alloc(M * K * 4 + 16)
        xb.upload(X, byte_offset=off)
        c0 = synth.activations(M, N, seed=92 + i).reshape(-1)
        for acc in (0, 1):
            ca, cb = backend.ctx.to_device(c0), backend.ctx.to_device(c0)
            assert L.trhip_gemm_q_actq_noalloc(h, w.h, 0, N, xb.addr(off), cb.addr(), M, K, acc) == 0, \
                L.trhip_last_error(h)
            assert L.trhip_gemm_q_actq(h, w.h, 0, N, xb.addr(off), ca.addr(), M, K, acc) == 0
            got = cb.download(np.float32, M * N)
            same_bits(got, ca.download(np.float32, M * N))
            if M * N * K <= 2e8:
                same_bits(got, O.quant_gemm_act(dt, M, N, K, X, raw, c0 if acc else None))
            for b in (ca, cb):
                b.free()
        xb.free()
        w.release()


@pytest.mark.parametrize("dt", [Q4K, Q6K])
def test_noalloc_padding_beyond_scratch(backend, dt):
    """33 rows whose row-major layout fits the scratch and whose 64 padded rows do not: a group of 32 rows and a single one."""
    M, N, K = 33, 40, 655360
    L = _lib.lib()
    raw = np.tile(synth.quant_weights(dt, N, 4096, seed=95, outliers=0.01).reshape(N, 1, -1), (1, K // 4096, 1)).reshape(-1)
    w = backend.FromQuantized(dt, raw, N, K)
    X = synth.activations(M, K, seed=96)
    X[31, 7], X[32, K - 1] = np.nan, np.inf
    xb, cb = backend.ctx.to_device(X), backend.ctx.alloc(M * N * 4)
    assert L.trhip_gemm_q_actq_noalloc(backend.ctx.h, w.h, 0, N, xb.addr(), cb.addr(), M, K, 0) == 0
    rows = [0, 1, 30, 31, 32]
    same_bits(cb.download(np.float32, M * N).reshape(M, N)[rows], O.quant_gemm_act(dt, len(rows), N, K, X[rows], raw))
    for b in (xb, cb):
        b.free()
    w.release()


@pytest.mark.parametrize("dt", [Q4K, Q6K])
@pytest.mark.parametrize("M", [1, 40])
def test_actq_captured_in_a_small_workspace(dt, M):
    """Captured on a context whose workspace (1 MB after a small call) holds the row-major layout but not the padded tiles'."""
    N, K = 64, 16384
    tb = QuantBackend(0)
    try:
        L = _lib.lib()
        raw = synth.quant_weights(dt, N, K, seed=97, outliers=0.01)
        w = tb.FromQuantized(dt, raw, N, K)
        X = synth.activations(M, K, seed=98)
        xb, cb, g = tb.ctx.to_device(X), tb.ctx.alloc(M * N * 4), ctypes.c_void_p()
        if M > 1:
            small = tb.FromQuantized(dt, raw[:raw.size // N // (K // 256)], 1, 256)
            tb.GemmActQuant(2, 1, 256, xb, small, cb, accumulate=False)
            small.release()
        assert L.trhip_graph_begin(tb.ctx.h) == 0
        try:
            tb.GemmActQuant(M, N, K, xb, w, cb, accumulate=False)
        finally:
            assert L.trhip_graph_end(tb.ctx.h, ctypes.byref(g)) == 0
        want = O.quant_gemm_act(dt, M, N, K, X, raw)
        for _ in range(3):
            cb.fill(0xFF)
            assert L.trhip_graph_launch(tb.ctx.h, g) == 0
            same_bits(cb.download(np.float32, M * N), want)
        assert L.trhip_graph_destroy(g) == 0
        for b in (xb, cb):
            b.free()
        w.release()
    finally:
        tb.close()


def test_noalloc_refuses_beyond_scratch(backend):
    L = _lib.lib()
    h = backend.ctx.h
    M, N, K = 4096, 8, 14336  # about 75 MB of scratch
    w = backend.FromQuantized(Q4K, synth.quant_weights(Q4K, N, K, seed=1, outliers=0.01), N, K)
    xb, cb = backend.ctx.alloc(M * K * 4), backend.ctx.alloc(M * N * 4)
    assert L.trhip_gemm_q_actq_noalloc(h, w.h, 0, N, xb.addr(), cb.addr(), M, K, 0) == 1
    assert b"scratch" in L.trhip_last_error(h)
    for b in (xb, cb):
        b.free()
    w.release()
