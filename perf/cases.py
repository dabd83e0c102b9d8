"""Performance cases of the MoE-FFN path: what a user of this library has it do.

Every case goes through the public entry points (qw3_amd.ds3 and the C ABI
behind it) on one Qwen3-30B-A3B-shaped layer or a small relative of it:

  layer    one MoE layer on the T tokens of a prefill chunk or of a decode
           batch, output zeroed first as the engine does (moe_ffn_batch)
  stack    a decode step: T streams through several layers' FFN blocks (norm,
           MoE, residual, in place), captured once and replayed as one graph
  token    the engine's GPU-only decode of one token: norm, zero, moe_ffn with
           the expert offset table, residual add, then the wait
  dense    the quantised products beside the MoE: output head, projections,
           and the few-row products of the host-bucketed prefill

prepare() quantises N(0, 0.02) weights to GGUF blocks on the GPU and lays them
out in the library's buffers; exact() evaluates the same bytes in 64 bits with
plain torch.
"""
from __future__ import annotations

import ctypes as C
import math

import numpy as np
import torch

from qw3_amd import ds3
from qw3_amd._native import hip

Q4, Q6, Q8, F32 = ds3.TYPE_Q4_K, ds3.TYPE_Q6_K, ds3.TYPE_Q8_0, ds3.TYPE_F32
TYPES = {"Q4_K": Q4, "Q6_K": Q6, "Q8_0": Q8}
EPS = 1e-6
STD = 0.02
QWEN = {"embd": 2048, "ff": 768, "experts": 128, "used": 8}


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------

def _layer(name, tokens, weights="Q4_K_M", zipf=False, **shape):
    return {"name": name, "kind": "layer", "tokens": tokens, "weights": weights, "zipf": zipf, **QWEN, **shape}


def _stack(name, tokens, layers, weights="Q4_K_M", **shape):
    return {"name": name, "kind": "stack", "tokens": tokens, "layers": layers, "weights": weights, **QWEN, **shape}


def _dense(name, rows, n, k, weights):
    return {"name": name, "kind": "dense", "rows": rows, "n": n, "k": k, "weights": weights}


def listed():
    return [
        # the smallest call: one decode token through one layer, waited for, as the engine's GPU-only decode makes it
        {"name": "token", "kind": "token", "weights": "Q4_K_M", **QWEN},
        # single-stream decode: one token through a quarter of the 48 layers, replayed as a graph
        _stack("decode_1x12", 1, 12),
        # batched decode (several streams, or a speculative draft): the few-token kernels
        _stack("decode_8x6", 8, 6),
        # few tokens on an all-Q8_0 layer, router included
        _layer("layer_q8_4", 4, "Q8_0"),
        # a short prompt, or the ragged tail of a chunked one: just past the few-token kernels
        _layer("layer_37", 37),
        # a mid-sized chunk of an all-Q8_0 model
        _layer("layer_q8_256", 256, "Q8_0"),
        # the engine's prefill chunk, balanced routing: the headline workload
        _layer("layer_512", 512),
        # a large chunk with Zipf-skewed expert popularity: empty experts beside very full ones
        _layer("layer_zipf_2048", 2048, zipf=True),
        # a whole long prompt in one call, ragged, several bucketing chunks
        _layer("layer_6001", 6001),
        # the output head of every decoded token
        _dense("head_q6k", 1, 151936, 2048, "Q6_K"),
        # one expert's gate product in the engine's own host-bucketed prefill (gather, three of these, scatter)
        _dense("expert_rows_27", 27, 768, 2048, "Q4_K"),
        # a prefill projection of a 512-token chunk
        _dense("projection_512", 512, 4096, 2048, "Q4_K"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 1)))))))


def draw(rng):
    kind = rng.choice(("layer", "layer", "layer", "stack", "dense", "dense"))
    if kind == "dense":
        weights = rng.choice(("Q4_K", "Q6_K", "Q8_0"))
        k = rng.choice((512, 768, 1024, 2048, 4096))
        rows = _log_int(rng, 1, 600)
        n = _log_int(rng, 64, 8192)
        if rows >= 64 and rng.random() < 0.7:
            n = max(256, n // 256 * 256)           # a model's own projection widths
        if rows == 1:
            n *= 16                                # one token: the heads and decode projections
        n = max(64, min(n, (1 << 31) // (rows * k)))
        return {"kind": kind, "rows": rows, "n": n, "k": k, "weights": weights}
    shape = dict(QWEN)
    if rng.random() < 0.4:
        shape = {"embd": rng.choice((512, 1024, 2048)), "ff": rng.choice((256, 512, 768)),
                 "experts": rng.choice((32, 64, 128)), "used": rng.choice((4, 8))}
    weights = rng.choice(("Q4_K_M", "Q4_K_M", "Q8_0"))
    if kind == "stack":
        tokens = _log_int(rng, 1, 16)
        return {"kind": kind, "tokens": tokens, "layers": rng.randint(1, max(1, min(12, 48 // tokens))),
                "weights": weights, **shape}
    return {"kind": kind, "tokens": _log_int(rng, 1, 4000 if weights == "Q8_0" else 6000), "weights": weights,
            "zipf": weights != "Q8_0" and rng.random() < 0.4, **shape}


# ---------------------------------------------------------------------------
# GGUF blocks of fp32 weights, on the GPU (w: [..., K] float32 -> uint8 rows)
# ---------------------------------------------------------------------------

def _f16_bytes(v):
    return v.to(torch.float16).unsqueeze(-1).view(torch.uint8)


def _q4_k(w):
    b = w.reshape(-1, 8, 32)
    lo = b.amin(2).clamp(max=0)
    sc, mn = (b.amax(2) - lo) / 15, -lo
    d, dm = ((v.amax(1) / 63).to(torch.float16) for v in (sc, mn))
    df, dmf = d.float().unsqueeze(1), dm.float().unsqueeze(1)
    s = (sc / df.clamp(min=1e-12)).round().clamp(0, 63)
    m = (mn / dmf.clamp(min=1e-12)).round().clamp(0, 63)
    q = ((b + (dmf * m).unsqueeze(2)) / (df * s).clamp(min=1e-12).unsqueeze(2)).round().clamp(0, 15).to(torch.uint8)
    s, m = s.to(torch.uint8), m.to(torch.uint8)
    q = q.reshape(-1, 4, 2, 32)
    qs = (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(-1, 128)
    sb = torch.cat((s[:, :4] | ((s[:, 4:] >> 4) << 6), m[:, :4] | ((m[:, 4:] >> 4) << 6),
                    (s[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)), 1)
    return torch.cat((_f16_bytes(d), _f16_bytes(dm), sb, qs), 1)


def _q6_k(w):
    b = w.reshape(-1, 16, 16)
    a = b.abs().amax(2) / 31
    d = (a.amax(1) / 127).to(torch.float16)
    df = d.float().unsqueeze(1)
    s = (a / df.clamp(min=1e-12)).round().clamp(1, 127)
    q = ((b / (df * s).clamp(min=1e-12).unsqueeze(2)).round().clamp(-32, 31) + 32).to(torch.uint8)
    q = q.reshape(-1, 2, 4, 32)                                     # half, 32t + l
    lo, hi = q & 15, q >> 4
    ql = torch.stack((lo[:, :, 0] | (lo[:, :, 2] << 4), lo[:, :, 1] | (lo[:, :, 3] << 4)), 2).reshape(-1, 128)
    qh = (hi[:, :, 0] | (hi[:, :, 1] << 2) | (hi[:, :, 2] << 4) | (hi[:, :, 3] << 6)).reshape(-1, 64)
    return torch.cat((ql, qh, s.to(torch.int8).view(torch.uint8), _f16_bytes(d)), 1)


def _q8_0(w):
    b = w.reshape(-1, 32)
    d = (b.abs().amax(1) / 127).to(torch.float16)
    q = (b / d.float().clamp(min=1e-12).unsqueeze(1)).round().clamp(-127, 127).to(torch.int8)
    return torch.cat((_f16_bytes(d), q.view(torch.uint8)), 1)


_QUANT = {Q4: _q4_k, Q6: _q6_k, Q8: _q8_0}


def _f16_at(blocks, at):
    return blocks[:, at:at + 2].contiguous().view(torch.float16).double()


def _dequant(t, raw, cols):
    """float64 values [rows][cols] of uint8 blocks, by the format's definition."""
    per, nb = ds3.BLOCK[t]
    b = raw.reshape(-1, nb)
    if t == F32:
        return raw.contiguous().view(torch.float32).double().reshape(-1, cols)
    if t == Q8:
        return (_f16_at(b, 0) * b[:, 2:].contiguous().view(torch.int8).double()).reshape(-1, cols)
    if t == Q6:
        d, s = _f16_at(b, 208), b[:, 192:208].contiguous().view(torch.int8).double()
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
        q = torch.stack([((ql[:, :, t_ & 1] >> (4 * (t_ >> 1))) & 15) | (((qh >> (2 * t_)) & 3) << 4)
                         for t_ in range(4)], 2).double() - 32
        return (d.unsqueeze(2) * s.unsqueeze(2) * q.reshape(-1, 16, 16)).reshape(-1, cols)
    d, dm, sb = _f16_at(b, 0), _f16_at(b, 2), b[:, 4:16]
    s = torch.cat((sb[:, :4] & 63, (sb[:, 8:] & 15) | ((sb[:, :4] >> 6) << 4)), 1).double()
    m = torch.cat((sb[:, 4:8] & 63, (sb[:, 8:] >> 4) | ((sb[:, 4:8] >> 6) << 4)), 1).double()
    qs = b[:, 16:].reshape(-1, 4, 32)
    q = torch.stack((qs & 15, qs >> 4), 2).reshape(-1, 8, 32).double()
    return ((d * s).unsqueeze(2) * q - (dm * m).unsqueeze(2)).reshape(-1, cols)


# ---------------------------------------------------------------------------
# Inputs, from the seed alone
# ---------------------------------------------------------------------------

def _gen(seed, *what):
    h = int(seed) * 1000003 + 17
    for w in what:
        h = (h * 1000003 + int(w) + 1) % (1 << 62)
    return torch.Generator(device="cuda").manual_seed(h)


def _normal(gen, rows, cols, std=1.0):
    return torch.randn(rows, cols, generator=gen, device="cuda") * std


def _matrix(t, gen, rows, cols, out=None):
    """[rows][cols] of N(0, 0.02) as blocks, a slice of rows at a time."""
    rb = ds3.row_bytes(t, cols)
    raw = torch.empty(rows * rb, dtype=torch.uint8, device="cuda") if out is None else out
    step = max(1, (1 << 25) // cols)
    for r in range(0, rows, step):
        n = min(step, rows - r)
        raw[r * rb:(r + n) * rb] = _QUANT[t](_normal(gen, n, cols, STD)).reshape(-1)
    return raw


def _types(case):
    """gate/up, down and router types of the layer."""
    return (Q8, Q8, Q8) if case["weights"] == "Q8_0" else (Q4, Q6, F32)


def _zipf_bias(n):
    """Logit bias ln(rank^-1.2) over a fixed permutation of the experts."""
    rank = np.random.default_rng(7).permutation(n) + 1
    p = rank.astype(np.float64) ** -1.2
    return np.log(p / p.sum()).astype(np.float32)


def _router(case, seed, layer):
    e, k, t = case["experts"], case["embd"], _types(case)[2]
    w = _normal(_gen(seed, layer, 0), e, k, STD)
    if t != F32:
        return _QUANT[t](w).reshape(-1)
    if case.get("zipf"):
        w[:, k - 1] = torch.from_numpy(_zipf_bias(e)).cuda()
    return w.contiguous().view(torch.uint8).reshape(-1)


def _tokens(case, seed, tokens):
    x = _normal(_gen(seed, 99), tokens, case["embd"])
    if case.get("zipf"):
        x[:, -1] = 1.0                                              # the input the router's bias column meets
    return x


def _experts(case, seed, layer, put):
    """gate, up and down blocks of the layer; put(type, rows, cols) gives the place of one tensor (None: a new one)."""
    e, k, f = case["experts"], case["embd"], case["ff"]
    tg, td, _ = _types(case)
    return [_matrix(t, _gen(seed, layer, 1 + i), rows, cols, put(t, rows, cols))
            for i, (t, rows, cols) in enumerate(((tg, e * f, k), (tg, e * f, k), (td, e * k, f)))]


# ---------------------------------------------------------------------------
# The library's buffers
# ---------------------------------------------------------------------------

class _Memory:
    """A ds3 buffer's device memory for torch (a handle starts with its base address, size and offset)."""

    def __init__(self, buf, shape, typestr):
        self.buf = buf
        base, _, offset = C.cast(buf.handle, C.POINTER(C.c_uint64))[0:3]
        self.__cuda_array_interface__ = {"shape": tuple(shape), "typestr": typestr, "data": (base + offset, False),
                                         "version": 2}


def _tensor(buf, shape, typestr="<f4"):
    return torch.as_tensor(_Memory(buf, shape, typestr), device="cuda")


def _device(t):
    """A buffer holding the tensor's bytes."""
    b = ds3.Buffer.alloc(t.numel() * t.element_size())
    _tensor(b, (b.nbytes,), "|u1").copy_(t.contiguous().view(torch.uint8).reshape(-1))
    return b


def _device_layer(case, seed, layer):
    """(router, experts): the router imported read-only, as the engine imports its mapped weights."""
    bufs = []

    def put(t, rows, cols):
        bufs.append(ds3.Buffer.alloc(rows * ds3.row_bytes(t, cols)))
        return _tensor(bufs[-1], (bufs[-1].nbytes,), "|u1")

    _experts(case, seed, layer, put)
    tg, td, _ = _types(case)
    router = ds3.Buffer.from_mmap_array(_router(case, seed, layer).cpu().numpy())
    return router, ds3.ExpertTensors(*bufs, tg, tg, td, case["embd"], case["ff"])


# A program enqueues its layers between begin_batch and end_batch; only the
# token case waits in each pass, as the engine does for each decoded token.
_batch_open = False


def _batch(open_):
    global _batch_open
    if open_ and not _batch_open:
        _ok(hip().ds3_hip_begin_batch())
    elif _batch_open and not open_:
        hip().ds3_hip_end_batch()
    _batch_open = open_


def _ok(rc):
    if rc != 0:
        raise RuntimeError("a library call failed")


class _State:
    pass


def prepare(case, seed):
    ds3.init()
    _batch(False)
    s = _State()
    s.case = case
    globals()["_prepare_" + case["kind"]](s, case, seed)
    torch.cuda.synchronize()                                        # the inputs are written on torch's stream
    if case["kind"] == "stack":
        _capture(s, case)
    _batch(case["kind"] != "token")
    return s


def run(state):
    return globals()["_run_" + state.case["kind"]](state)


def _prepare_layer(s, case, seed):
    t, k, u = case["tokens"], case["embd"], case["used"]
    s.router, s.experts = _device_layer(case, seed, 0)
    s.x = _device(_tokens(case, seed, t))
    s.out, s.idx, s.scores = (ds3.Buffer.alloc(4 * n) for n in (t * k, t * u, t * u))
    s.outputs = {"out": _tensor(s.out, (t, k)), "indices": _tensor(s.idx, (t, u), "<i4"),
                 "scores": _tensor(s.scores, (t, u))}


def _run_layer(s):
    c = s.case
    s.out.zero()
    ds3.moe_ffn_batch(s.x, s.router, _types(c)[2], s.experts, s.out, c["tokens"], c["experts"], c["used"],
                      indices=s.idx, scores=s.scores)
    return s.outputs


def _prepare_stack(s, case, seed):
    t, k, u, n = case["tokens"], case["embd"], case["used"], case["layers"]
    s.layers = [_device_layer(case, seed, i) for i in range(n)]
    s.norm = _device(_gain(case, seed))
    s.x = _device(_tokens(case, seed, t))
    s.hidden, s.idx = ds3.Buffer.alloc(4 * t * k), ds3.Buffer.alloc(4 * n * t * u)
    s.idx_of = [s.idx.view(4 * i * t * u, 4 * t * u) for i in range(n)]
    s.outputs = {"hidden": _tensor(s.hidden, (t, k)), "indices": _tensor(s.idx, (n, t, u), "<i4")}


def _gain(case, seed):
    return 1.0 + _normal(_gen(seed, 98), 1, case["embd"], STD)


def _stack_calls(s, case):
    _ok(hip().ds3_hip_buffer_copy_f32(s.x, s.hidden, s.x.nbytes))
    for (router, experts), idx in zip(s.layers, s.idx_of):
        ds3.moe_block(s.hidden, s.norm, EPS, router, _types(case)[2], experts, case["tokens"], case["experts"],
                      case["used"], indices=idx)


def _capture(s, case):
    _stack_calls(s, case)                                           # the workspace is there before the capture
    with ds3.Graph() as s.graph:
        _stack_calls(s, case)


def _run_stack(s):
    s.graph.launch()
    return s.outputs


def _prepare_token(s, case, seed):
    e, k, f = case["experts"], case["embd"], case["ff"]
    s.router, s.experts = _device_layer(case, seed, 0)
    strides = s.experts.strides
    table = np.stack([np.arange(e, dtype=np.uint64) * np.uint64(rows * st)
                      for rows, st in zip((f, f, k), strides)], 1)
    s.table = ds3.Buffer.from_array(table)
    s.norm, s.hidden = _device(_gain(case, seed)), _device(_tokens(case, seed, 1))
    s.xn, s.out, s.y, s.scratch = (ds3.Buffer.alloc(4 * n) for n in (k, k, k, max(k, case["used"] * f)))
    s.logits = ds3.Buffer.alloc(4 * e)
    s.outputs = {"hidden": _tensor(s.y, (1, k)), "logits": _tensor(s.logits, (1, e))}


def _run_token(s):
    c, k = s.case, s.case["embd"]
    _ok(hip().ds3_hip_begin_batch())
    ds3.rms_norm(s.hidden, s.norm, s.xn, k, 1, EPS)
    s.out.zero()
    ds3.moe_ffn(s.xn, s.router, _types(c)[2], s.experts, s.out, s.logits, c["experts"], c["used"], scratch=s.scratch,
                expert_offsets=s.table)
    _ok(hip().ds3_hip_vec_add(s.out, s.hidden, s.y, k))
    hip().ds3_hip_end_batch()
    return s.outputs


def _prepare_dense(s, case, seed):
    t, m, n, k = TYPES[case["weights"]], case["rows"], case["n"], case["k"]
    s.w = ds3.Buffer.alloc(n * ds3.row_bytes(t, k))
    _matrix(t, _gen(seed, 1), n, k, _tensor(s.w, (s.w.nbytes,), "|u1"))
    s.a = _device(_normal(_gen(seed, 2), m, k))
    s.c = ds3.Buffer.alloc(4 * m * n)
    s.outputs = {"c": _tensor(s.c, (m, n))}


def _run_dense(s):
    c = s.case
    t, m, n, k = TYPES[c["weights"]], c["rows"], c["n"], c["k"]
    if m == 1:
        _ok(hip().ds3_hip_vec_matmul_quantized(s.a, s.w, s.c, k, n, ds3.row_bytes(t, k), t))
    else:
        _ok(hip().ds3_hip_matmul_quantized_batch(s.a, s.w, s.c, m, n, k, ds3.row_bytes(t, k), 0, t))
    return s.outputs


# ---------------------------------------------------------------------------
# Work, tolerance, 64-bit results
# ---------------------------------------------------------------------------

def _distinct(case, tokens):
    """Experts that `tokens` tokens are expected to choose between them (sampled logits of the inputs' distribution)."""
    e, u = case["experts"], case["used"]
    std = STD * math.sqrt(case["embd"])
    z = np.random.default_rng(3).standard_normal((tokens, e)) * std
    if case.get("zipf"):
        z += _zipf_bias(e)
    return len(np.unique(np.argpartition(-z, u - 1, axis=1)[:, :u]))


def work(case):
    if case["kind"] == "dense":
        m, n, k = case["rows"], case["n"], case["k"]
        return {"bytes": n * ds3.row_bytes(TYPES[case["weights"]], k) + 4 * m * (n + k), "flops": 2 * m * n * k}
    t, layers = case.get("tokens", 1), case.get("layers", 1)
    e, k, f, u = case["experts"], case["embd"], case["ff"], case["used"]
    tg, td, tr = _types(case)
    expert = 2 * f * ds3.row_bytes(tg, k) + k * ds3.row_bytes(td, f)
    return {"bytes": layers * (_distinct(case, t) * expert + e * ds3.row_bytes(tr, k)) + 2 * 4 * t * k,
            "flops": layers * 2 * t * k * (e + 3 * u * f)}


def _fp16_operands(case):
    """Whether the products take fp16 operands, as the header states: the prefill kernels (from 17 tokens), and dense
    products of 64 rows up of the shapes named there."""
    if case["kind"] == "dense":
        return case["rows"] >= 64 and case["k"] % 512 == 0 and case["n"] % 256 == 0
    return case.get("tokens", 1) >= 17


def tolerance(case):
    # Operands in fp16 (x, weights, h, y): 3 to 6e-4 off the 64-bit result.  fp32
    # throughout: 1e-7 to 1.4e-6 (sums of 2048 terms, then of 768).  About four times that.
    if _fp16_operands(case):
        return {"rel": 2e-3, "max": 2e-2, "differ": 0.0}
    return {"rel": 6e-6, "max": 1e-4, "differ": 0.0}


def _moe64(case, x, router, experts):
    """(output, logits, weights) of the layer on float64 rows x."""
    e, k, f, u = case["experts"], case["embd"], case["ff"], case["used"]
    tg, td, tr = _types(case)
    logits = x @ _dequant(tr, router, k).t()
    w, idx = torch.topk(torch.softmax(logits, 1), u, dim=1)
    w = w / w.sum(1, keepdim=True)
    out = torch.zeros_like(x)
    for i in range(e):
        t, j = torch.nonzero(idx == i, as_tuple=True)
        if t.numel() == 0:
            continue
        g, up, d = (_dequant(ty, raw[i * rows * ds3.row_bytes(ty, c):(i + 1) * rows * ds3.row_bytes(ty, c)], c)
                    for ty, raw, rows, c in zip((tg, tg, td), experts, (f, f, k), (k, k, f)))
        h = torch.nn.functional.silu(x[t] @ g.t()) * (x[t] @ up.t())
        out.index_add_(0, t, (h @ d.t()) * w[t, j].unsqueeze(1))
    return out, logits, w


def _norm64(x, gain):
    return x / torch.sqrt((x * x).mean(1, keepdim=True) + EPS) * gain


def exact(case, seed):
    if case["kind"] == "dense":
        t, m, n, k = TYPES[case["weights"]], case["rows"], case["n"], case["k"]
        raw, rb = _matrix(t, _gen(seed, 1), n, k), ds3.row_bytes(t, k)
        a = _normal(_gen(seed, 2), m, k).double()
        return {"c": torch.cat([a @ _dequant(t, raw[r * rb:(r + 8192) * rb], k).t() for r in range(0, n, 8192)], 1)}
    x = _tokens(case, seed, case.get("tokens", 1)).double()
    gain = _gain(case, seed).double()
    for i in range(case.get("layers", 1)):
        xn = x if case["kind"] == "layer" else _norm64(x, gain)
        experts = _experts(case, seed, i, lambda *_: None)
        out, logits, w = _moe64(case, xn, _router(case, seed, i), experts)
        if case["kind"] == "layer":
            return {"out": out, "indices": None, "scores": w}
        x = x + out
    if case["kind"] == "token":
        return {"hidden": x, "logits": logits}
    return {"hidden": x, "indices": None}
