"""The work this library does for a program that runs a quantized language model, as cases to time and to compare.

Every case goes through the operator interface (tcb_amd.QuantBackend) on weights in the four GGUF block formats. Sizes
are those of the benchmark and the tests (hidden 4096, FFN 14336, 1024-row k / v projections, a 128256-row q6_k table),
and draw() spreads them over the range between the smallest projections and the largest prompts, ragged ones included.

exact() restates the operators in float64 from the block formats alone.
"""
import ctypes
import math

import torch

from tcb_amd import MODE_EXACT, MODE_FAST, Q4, Q4K, Q6K, Q8, QuantBackend, _lib

DT = {"q8_0": Q8, "q4_0": Q4, "q4_k": Q4K, "q6_k": Q6K}
BLOCK = {"q8_0": (32, 34), "q4_0": (32, 18), "q4_k": (256, 144), "q6_k": (256, 210)}  # elements, bytes
IO = {"f32": (_lib.F32, torch.float32), "f16": (_lib.F16, torch.float16), "bf16": (_lib.BF16, torch.bfloat16)}
HEAD_ROWS = 128256
# multiply-adds of the largest drawn product: 512 rows through a 14336 x 4096 layer
MOST_MACS = 512 * 14336 * 4096
DEV = "cuda:0"


def listed():
    return [
        # the smallest call of a decode step: one token through a k or v projection, where the launch counts
        dict(name="kv token fast", kind="gemm", dtype="q4_k", N=1024, K=4096, M=1, fast=True, io="f32"),
        # a token step of four merged layers and the output head, replayed as a graph: chat at batch 1
        dict(name="step token", kind="step", batch=1, layers=4, hidden=4096, kv=1024, ffn=14336, head=HEAD_ROWS),
        # the same step for sixteen sequences at once: serving
        dict(name="step batch 16", kind="step", batch=16, layers=4, hidden=4096, kv=1024, ffn=14336, head=HEAD_ROWS),
        # the default mode's decode GEMV on the widest rows: an FFN down projection kept in q6_k
        dict(name="down token exact", kind="gemm", dtype="q6_k", N=4096, K=14336, M=1, fast=False, io="f32"),
        # a few sequences together in the default mode, with 16-bit activations: merged q/k/v in q8_0
        dict(name="qkv 5 rows exact bf16", kind="gemm", dtype="q8_0", N=6144, K=4096, M=5, fast=False, io="bf16"),
        # a short prompt of odd length in the default mode: an attention output projection
        dict(name="prompt 77 exact", kind="gemm", dtype="q4_k", N=4096, K=4096, M=77, fast=False, io="f32"),
        # an ordinary prompt chunk in fast mode: the gate or up projection
        dict(name="prompt 512 fast", kind="gemm", dtype="q4_k", N=14336, K=4096, M=512, fast=True, io="f32"),
        # a prompt of a q8_0 model in fast mode: the down projection
        dict(name="prompt 300 fast q8_0", kind="gemm", dtype="q8_0", N=4096, K=14336, M=300, fast=True, io="f32"),
        # quantized activations switched on for a whole chat: one decoded token, gate or up projection
        dict(name="actq token", kind="actq", dtype="q4_k", N=14336, K=4096, M=1, fast=False),
        # and the longest prompt chunk of it
        dict(name="actq prompt 2048", kind="actq", dtype="q4_k", N=14336, K=4096, M=2048, fast=False),
        # a ragged prompt chunk through a q6_k down projection
        dict(name="actq prompt 130 q6_k", kind="actq", dtype="q6_k", N=4096, K=14336, M=130, fast=False),
        # the token embedding of a prompt from the q6_k table
        dict(name="embed 512", kind="embed", dtype="q6_k", N=HEAD_ROWS, K=4096, M=512),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["gemm", "gemm", "gemm", "swiglu", "actq", "actq", "step", "embed", "open"])
    if kind == "step":
        hidden = 256 * rng.randint(4, 16)
        return dict(kind=kind, batch=rng.choice([1, 1, rng.randint(2, 16)]), layers=rng.randint(1, 4), hidden=hidden,
                    kv=128 * rng.randint(2, 8), ffn=256 * rng.randint(12, 56), head=_log_int(rng, 8000, HEAD_ROWS))
    dtype = rng.choice(["q4_k", "q6_k"] if kind == "swiglu" else ["q8_0", "q4_0", "q4_k", "q6_k"])
    if kind == "actq" and dtype == "q8_0":  # not an act-quant format
        dtype = "q4_k"
    unit = BLOCK[dtype][0]
    K = max(256, _log_int(rng, 512, 16384) // 256 * 256)
    if unit == 32 and rng.random() < 0.3:  # a ragged tail behind the last 256 elements
        K += 32 * rng.randint(1, 7)
    N = _log_int(rng, 256, 32768)
    if rng.random() < 0.6:
        N = max(256, N // 128 * 128)
    if kind == "embed":
        return dict(kind=kind, dtype=dtype, N=N, K=K, M=_log_int(rng, 1, 2048))
    if kind == "open":
        return dict(kind=kind, dtype=dtype, N=N, K=K, M=1)
    M = min(_log_int(rng, 1, 2048), max(1, MOST_MACS // (N * K)))
    if rng.random() < 0.3:
        M = 1
    fast = rng.random() < 0.5
    if kind == "swiglu":
        return dict(kind=kind, dtype=dtype, N=2 * (N // 2), K=K, M=M, fast=fast)
    if kind == "actq":
        return dict(kind=kind, dtype=dtype, N=N, K=K, M=M, fast=fast)
    return dict(kind=kind, dtype=dtype, N=N, K=K, M=M, fast=fast, io=rng.choice(["f32", "f32", "bf16", "f16"]))


# ---- weights: N(0, 0.02) with one in a hundred scaled by ten, encoded into GGUF blocks on the GPU -------------------

def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(int(seed) & 0x7FFFFFFF)
    return g


def _f16_bytes(v):
    return v.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _div(a, b):
    return torch.where(b != 0, a / torch.where(b != 0, b, torch.ones_like(b)), torch.zeros_like(a))


def _enc_q8_0(b):
    d = (b.abs().amax(2) / 127).to(torch.float16).float()
    q = torch.round(_div(b, d.unsqueeze(2).expand_as(b))).clamp_(-127, 127).to(torch.int8)
    return torch.cat([_f16_bytes(d), q.view(torch.uint8)], 2)


def _enc_q4_0(b):
    peak = b.gather(2, b.abs().argmax(2, keepdim=True)).squeeze(2)
    d = (peak / -8).to(torch.float16).float()
    q = torch.floor(_div(b, d.unsqueeze(2).expand_as(b)) + 8.5).clamp_(0, 15).to(torch.uint8)
    return torch.cat([_f16_bytes(d), q[..., :16] | (q[..., 16:] << 4)], 2)


def _enc_q4_k(b):
    R, nb, _ = b.shape
    s = b.view(R, nb, 8, 32)
    low = s.amin(3).clamp(max=0)
    scale, mins = (s.amax(3) - low) / 15, -low
    d = (scale.amax(2) / 63).to(torch.float16).float()
    dmin = (mins.amax(2) / 63).to(torch.float16).float()
    sc = torch.round(_div(scale, d.unsqueeze(2).expand_as(scale))).clamp_(0, 63)
    mn = torch.round(_div(mins, dmin.unsqueeze(2).expand_as(mins))).clamp_(0, 63)
    d1, m1 = (d.unsqueeze(2) * sc).unsqueeze(3).expand_as(s), (dmin.unsqueeze(2) * mn).unsqueeze(3)
    q = torch.round(_div(s + m1, d1)).clamp_(0, 15).to(torch.uint8).view(R, nb, 4, 2, 32)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    packed = torch.cat([sc[..., :4] | ((sc[..., 4:] >> 4) << 6), mn[..., :4] | ((mn[..., 4:] >> 4) << 6),
                        (sc[..., 4:] & 15) | ((mn[..., 4:] & 15) << 4)], 2)
    qs = (q[..., 0, :] | (q[..., 1, :] << 4)).view(R, nb, 128)
    return torch.cat([_f16_bytes(d), _f16_bytes(dmin), packed, qs], 2)


def _enc_q6_k(b):
    R, nb, _ = b.shape
    s = b.view(R, nb, 16, 16)
    scale = s.gather(3, s.abs().argmax(3, keepdim=True)).squeeze(3) / -32
    d = (scale.abs().amax(2) / 127).to(torch.float16).float()
    sc = torch.round(_div(scale, d.unsqueeze(2).expand_as(scale))).clamp_(-127, 127)
    step = (d.unsqueeze(2) * sc).unsqueeze(3).expand_as(s)
    q = (torch.round(_div(s, step)).clamp_(-32, 31) + 32).to(torch.uint8).view(R, nb, 2, 4, 32)
    ql = torch.stack([(q[..., 0, :] & 15) | ((q[..., 2, :] & 15) << 4),
                      (q[..., 1, :] & 15) | ((q[..., 3, :] & 15) << 4)], 3).view(R, nb, 128)
    top = q >> 4
    qh = (top[..., 0, :] | (top[..., 1, :] << 2) | (top[..., 2, :] << 4) | (top[..., 3, :] << 6)).view(R, nb, 64)
    return torch.cat([ql, qh, sc.to(torch.int8).view(torch.uint8), _f16_bytes(d)], 2)


_ENCODE = {"q8_0": _enc_q8_0, "q4_0": _enc_q4_0, "q4_k": _enc_q4_k, "q6_k": _enc_q6_k}


def _row_chunks(N, K):
    step = max(1, (1 << 25) // K)
    return [(r, min(N, r + step)) for r in range(0, N, step)]


def _raw_blocks(dtype, N, K, seed):
    """Encoded rows in file order, as a uint8 GPU tensor [N, blocks, bytes]."""
    unit, size = BLOCK[dtype]
    out = torch.empty((N, K // unit, size), dtype=torch.uint8, device=DEV)
    g = _gen(seed)
    for r0, r1 in _row_chunks(N, K):
        w = torch.randn((r1 - r0, K // unit, unit), generator=g, device=DEV) * 0.02
        w[torch.rand(w.shape, generator=g, device=DEV) < 0.01] *= 10
        out[r0:r1] = _ENCODE[dtype](w)
    return out


def _f16_at(raw, at):
    return raw[..., at:at + 2].contiguous().view(torch.float16).double()


def _decode(dtype, raw):
    """float64 [rows, K] of encoded rows [rows, blocks, bytes]."""
    R, nb, _ = raw.shape
    if dtype == "q8_0":
        w = _f16_at(raw, 0) * raw[..., 2:].contiguous().view(torch.int8).double()
    elif dtype == "q4_0":
        q = raw[..., 2:]
        w = _f16_at(raw, 0) * (torch.cat([q & 15, q >> 4], 2).double() - 8)
    elif dtype == "q4_k":
        s = raw[..., 4:16]
        sc = torch.cat([s[..., :4] & 63, (s[..., 8:] & 15) | ((s[..., :4] >> 6) << 4)], 2).double()
        mn = torch.cat([s[..., 4:8] & 63, (s[..., 8:] >> 4) | ((s[..., 4:8] >> 6) << 4)], 2).double()
        q = raw[..., 16:].view(R, nb, 4, 32)
        q = torch.stack([q & 15, q >> 4], 3).view(R, nb, 8, 32).double()
        w = (_f16_at(raw, 0) * sc).unsqueeze(3) * q - (_f16_at(raw, 2) * mn).unsqueeze(3)
    else:
        ql, qh = raw[..., :128].view(R, nb, 2, 2, 32), raw[..., 128:192].view(R, nb, 2, 32)
        q = torch.stack([(ql[..., 0, :] & 15) | ((qh & 3) << 4), (ql[..., 1, :] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[..., 0, :] >> 4) | (((qh >> 4) & 3) << 4), (ql[..., 1, :] >> 4) | ((qh >> 6) << 4)], 3)
        sc = raw[..., 192:208].contiguous().view(torch.int8).double()
        w = (_f16_at(raw, 208) * sc).unsqueeze(3) * (q.reshape(R, nb, 16, 16).double() - 32)
    return w.reshape(R, -1)


# ---- inputs --------------------------------------------------------------------------------------------------------

_backend = []


def _tb():
    if not _backend:
        _backend.append(QuantBackend(0))
    return _backend[0]


class State:
    """What a program holds between calls; releases its stores and graph with itself."""

    def __init__(self, case):
        self.case, self.stores, self.graph, self.out = case, [], None, None

    def store(self, dtype, N, K, seed):
        w = _tb().FromQuantized(DT[dtype], _raw_blocks(dtype, N, K, seed).reshape(-1).cpu().numpy(), N, K)
        self.stores.append(w)
        return w

    def __del__(self):
        _tb().ctx.sync()
        if self.graph is not None:
            _lib.lib().trhip_graph_destroy(self.graph)
        for w in self.stores:
            w.release()


def _activations(shape, seed, dtype=torch.float32):
    return torch.randn(shape, generator=_gen(seed), device=DEV).to(dtype)


def _step_layers(case):
    """(dtype, N, K) of a layer's merged weights: [q | k | v], o, [gate | up], down."""
    h, f = case["hidden"], case["ffn"]
    return [("q4_k", h + 2 * case["kv"], h), ("q4_k", h, h), ("q4_k", 2 * f, h), ("q4_k", h, f)]


def _step_calls(s):
    tb, case, b = _tb(), s.case, s.case["batch"]
    for layer, x, att, outs in s.layers:
        qkv, o, gu, down = layer
        tb.GemmSet(b, qkv.N, qkv.K, x.data_ptr(), qkv, outs[0].data_ptr(), mode=MODE_FAST)
        tb.GemmSet(b, o.N, o.K, att.data_ptr(), o, outs[1].data_ptr(), mode=MODE_FAST)
        tb.GemmSwiGLU(b, gu.K, x.data_ptr(), gu, outs[2].data_ptr(), mode=MODE_FAST)
        tb.GemmSet(b, down.N, down.K, outs[2].data_ptr(), down, outs[3].data_ptr(), mode=MODE_FAST)
    tb.GemmSet(b, s.head.N, s.head.K, s.x.data_ptr(), s.head, s.logits.data_ptr(), mode=MODE_FAST)


def _prepare_step(case, seed):
    s, b, h = State(case), case["batch"], case["hidden"]
    s.layers, s.out = [], []
    for i in range(case["layers"]):
        shapes = _step_layers(case)
        layer = [s.store(dt, n, k, seed * 1009 + 16 * i + j) for j, (dt, n, k) in enumerate(shapes)]
        x, att = _activations((b, h), seed * 1013 + 2 * i), _activations((b, h), seed * 1013 + 2 * i + 1)
        outs = [torch.empty((b, n // 2 if j == 2 else n), device=DEV) for j, (_, n, _) in enumerate(shapes)]
        s.layers.append((layer, x, att, outs))
        s.out.append(outs)
    s.head = s.store("q6_k", case["head"], h, seed * 1009 + 999)
    s.x, s.logits = _activations((b, h), seed * 1013 + 999), torch.empty((b, case["head"]), device=DEV)
    s.out.append(s.logits)
    torch.cuda.synchronize()
    _step_calls(s)  # sizes the workspace before the capture
    L, ctx = _lib.lib(), _tb().ctx
    ctx.sync()
    if L.trhip_graph_begin(ctx.h):
        raise RuntimeError("graph begin")
    _step_calls(s)
    graph = ctypes.c_void_p()
    if L.trhip_graph_end(ctx.h, ctypes.byref(graph)):
        raise RuntimeError("graph end")
    s.graph = graph
    return s


def prepare(case, seed):
    if case["kind"] == "step":
        return _prepare_step(case, seed)
    s = State(case)
    N, K, M = case["N"], case["K"], case["M"]
    s.w = s.store(case["dtype"], N, K, seed * 1009)
    if case["kind"] == "embed":
        s.idx = torch.randint(0, N, (M,), generator=_gen(seed * 1013), device=DEV).cpu().numpy()
        s.out = torch.empty((M, K), device=DEV)
    elif case["kind"] == "open":
        s.out = torch.empty((N, K), device=DEV)
    else:
        t = IO[case.get("io", "f32")][1]
        s.x = _activations((M, K), seed * 1013, t)
        s.out = torch.empty((M, N // 2 if case["kind"] == "swiglu" else N), device=DEV, dtype=t)
    torch.cuda.synchronize()
    return s


def run(s):
    case, tb = s.case, _tb()
    kind = case["kind"]
    if kind == "step":
        if _lib.lib().trhip_graph_launch(tb.ctx.h, s.graph):
            raise RuntimeError("graph launch")
        return s.out
    if kind == "embed":
        tb.Embedding(s.out.data_ptr(), s.w, s.idx)
        return s.out
    if kind == "open":
        tb.OpenQuant(s.out.data_ptr(), s.w)
        return s.out
    mode = MODE_FAST if case["fast"] else MODE_EXACT
    M, N, K = case["M"], case["N"], case["K"]
    if kind == "swiglu":
        tb.GemmSwiGLU(M, K, s.x.data_ptr(), s.w, s.out.data_ptr(), mode=mode)
    elif kind == "actq":
        tb.GemmActQuant(M, N, K, s.x.data_ptr(), s.w, s.out.data_ptr(), accumulate=False, mode=mode)
    elif case["io"] == "f32":
        tb.GemmSet(M, N, K, s.x.data_ptr(), s.w, s.out.data_ptr(), mode=mode)
    else:
        io = IO[case["io"]][0]
        tb.GemmTyped(M, N, K, s.x.data_ptr(), io, s.w, s.out.data_ptr(), io, mode=mode)
    return s.out


def _weight_bytes(dtype, N, K):
    unit, size = BLOCK[dtype]
    return N * (K // unit) * size


def work(case):
    """Weights, activations and outputs once; two operations per weight and row."""
    if case["kind"] == "step":
        b, nbytes, flops = case["batch"], 0, 0
        shapes = _step_layers(case) * case["layers"] + [("q6_k", case["head"], case["hidden"])]
        for dt, n, k in shapes:
            nbytes += _weight_bytes(dt, n, k) + 4 * b * (n + k)
            flops += 2 * b * n * k
        return {"bytes": nbytes, "flops": flops}
    N, K, M = case["N"], case["K"], case["M"]
    if case["kind"] == "embed":
        return {"bytes": _weight_bytes(case["dtype"], M, K) + 8 * M + 4 * M * K, "flops": M * K}
    if case["kind"] == "open":
        return {"bytes": _weight_bytes(case["dtype"], N, K) + 4 * N * K, "flops": N * K}
    e = 4 if case.get("io", "f32") == "f32" else 2
    n_out = N // 2 if case["kind"] == "swiglu" else N
    return {"bytes": _weight_bytes(case["dtype"], N, K) + e * M * (K + n_out), "flops": 2 * M * N * K}


def tolerance(case):
    # Exact mode, embedding and dequantization promise the bits of one fixed order of operations.
    if case["kind"] in ("embed", "open") or (case["kind"] != "step" and not case["fast"]):
        return "exact"
    if case.get("io", "f32") != "f32":  # one rounding to 16 bits on top: a flipped last bit here and there
        return {"rel": 1e-4, "max": 2e-3} if case["io"] == "f16" else {"rel": 3e-4, "max": 1.6e-2}
    # Measured against float64: 0.2e-6 to 0.9e-6 for one product, 1.0e-6 for the two in a row of a step's FFN.
    return {"rel": 4e-6, "max": 8e-5}


# ---- the same operators in float64 ------------------------------------------------------------------------------------

def _product(dtype, N, K, seed, x):
    raw, out = _raw_blocks(dtype, N, K, seed), torch.empty((x.shape[0], N), dtype=torch.float64, device=DEV)
    x = x.double()
    for r0, r1 in _row_chunks(N, K):
        out[:, r0:r1] = x @ _decode(dtype, raw[r0:r1]).t()
    return out


def _swiglu(gu):
    g, u = gu.chunk(2, 1)
    return g * torch.sigmoid(g) * u


def _quantized(x, blk):
    """The activations the act-quant operator multiplies: per block of a row d = max|x| / 127 and whole codes."""
    b = x.view(x.shape[0], -1, blk)
    peak = b.abs().amax(2, keepdim=True)
    codes = torch.round(b * _div(torch.full_like(peak, 127), peak)).clamp_(-127, 127)
    return (codes.double() * (peak / 127).double()).view(x.shape)


def exact(case, seed):
    if case["kind"] == "step":
        out, b, h = [], case["batch"], case["hidden"]
        for i in range(case["layers"]):
            x, att = _activations((b, h), seed * 1013 + 2 * i), _activations((b, h), seed * 1013 + 2 * i + 1)
            ys = []
            for j, (dt, n, k) in enumerate(_step_layers(case)):
                y = _product(dt, n, k, seed * 1009 + 16 * i + j, (x, att, x, ys[-1] if ys else x)[j])
                ys.append(_swiglu(y) if j == 2 else y)
            out.append(ys)
        out.append(_product("q6_k", case["head"], h, seed * 1009 + 999, _activations((b, h), seed * 1013 + 999)))
        return out
    N, K, M = case["N"], case["K"], case["M"]
    if case["kind"] in ("embed", "open"):
        raw = _raw_blocks(case["dtype"], N, K, seed * 1009)
        if case["kind"] == "embed":
            raw = raw[torch.randint(0, N, (M,), generator=_gen(seed * 1013), device=DEV)]
        return torch.cat([_decode(case["dtype"], raw[r0:r1]) for r0, r1 in _row_chunks(raw.shape[0], K)])
    x = _activations((M, K), seed * 1013, IO[case.get("io", "f32")][1])
    if case["kind"] == "actq":
        x = _quantized(x, BLOCK[case["dtype"]][0])
    y = _product(case["dtype"], N, K, seed * 1009, x)
    return _swiglu(y) if case["kind"] == "swiglu" else y
