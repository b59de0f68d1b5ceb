"""The work this library does for its users, as cases that can be timed and checked.

A case is one pass through the public entry points over a few layers of a model shape:

  decode        pqa_decode of every layer at one position (a token of a serving loop whose
                projections run elsewhere); with "graph", the same step captured once with
                pqa_decode_noalloc and replayed;
  prefill       pqa_prefill of every layer for a prompt chunk, on an empty cache or behind a
                history (the next turn of a chat, a prompt after a loaded .kvc file);
  token_block   pqa_attention_block: one token from the normed input to the residual stream,
                GGUF weights included; with "host", PicoAttention.attention_block on numpy
                arrays, as the CPU forward loop calls it;
  prompt_block  pqa_prefill_block: the same for a prompt chunk; with "host" on numpy arrays.

Shapes are those of the benchmark and the tests; positions run from 0 to 131071, prompts from
2 to 2048 tokens. Inputs are q, k, v and normed rows ~N(0, 1), a cache of N(0, 1) rows (with
"outliers", 1 % of them times 8), norm weights near 1 and weights of about 1 / sqrt(width).

exact() is the same block in 64-bit floats from the same inputs, weights dequantized by the GGUF
formulas and the new K/V rows rounded to the cache's fp16.
"""
import contextlib
import ctypes as C
import math

import numpy as np
import torch

from picolm_qwen_amd import PicoAttention
from picolm_qwen_amd._lib import check, lib
from picolm_qwen_amd.hipgraph import Graph

F32, F16, Q8_0, Q4_K, Q6_K = 1, 2, 9, 13, 15
NEOX, BLOCK8 = 0, 1

# name: query heads, KV heads, head size, RoPE pairing and base, QK-norm, input width, q/k/v biases
MODELS = {
    "tinyllama": (32, 4, 64, BLOCK8, 1e4, False, 2048, False),
    "qwen2.5_0.5b": (14, 2, 64, NEOX, 1e6, False, 896, True),
    "qwen3_1.7b": (16, 8, 128, NEOX, 1e6, True, 2048, False),
    "qwen3_4b": (32, 8, 128, NEOX, 1e6, True, 2560, False),
    "qwen3_8b": (32, 8, 128, NEOX, 1e6, True, 4096, False),
    # head sizes outside 64 and 128, as the tests run them
    "hd80": (16, 4, 80, NEOX, 1e6, True, 1280, False),
    "hd96": (32, 8, 96, BLOCK8, 1e4, True, 3072, False),
    "hd256": (8, 2, 256, NEOX, 1e6, True, 2048, False),
}


def _case(name, op, model, layers, pos, n_tok=1, weights="", outliers=False, graph=False, host=False, exact_kv=True):
    c = {"op": op, "model": model, "layers": layers, "pos": pos, "n_tok": n_tok, "weights": weights,
         "outliers": outliers, "graph": graph, "host": host, "exact_kv": exact_kv}
    return dict(c, name=name) if name else c


def listed():
    return [
        # a short chat on a small model: every layer of a token, launch and latency bound
        _case("decode_small_512", "decode", "tinyllama", 22, 511),
        # a serving loop's captured step in the middle of a conversation, at a ragged position
        _case("decode_graph_1900", "decode", "qwen2.5_0.5b", 24, 1899, graph=True),
        # a long document
        _case("decode_32k", "decode", "qwen3_1.7b", 8, 32767),
        # the longest context, with outlier rows: the benchmark's headline shape
        _case("decode_131k", "decode", "qwen3_8b", 4, 131071, outliers=True),
        # a head size outside 64 and 128
        _case("decode_hd96_9000", "decode", "hd96", 8, 8999),
        # a whole prompt in one pass
        _case("prefill_2048", "prefill", "qwen3_4b", 4, 0, 2048),
        # the next turn of a chat: a ragged chunk behind a long history
        _case("prefill_turn_300_at_12000", "prefill", "qwen3_4b", 4, 12000, 300),
        # a prompt at another head size
        _case("prefill_hd96_700", "prefill", "hd96", 2, 0, 700),
        # one token of a quantized model through the attention half of its layers
        _case("token_block_q4k_4096", "token_block", "qwen3_8b", 4, 4095, weights="q4_k_m"),
        # the CPU forward loop with this library in its attention half (host vectors, a sync per layer)
        _case("token_block_host_q8_300", "token_block", "qwen2.5_0.5b", 8, 299, weights="q8_0", host=True),
        # a short chat prompt through the attention half of a layer, cache rows bit-exact
        _case("prompt_block_75", "prompt_block", "qwen3_4b", 4, 0, 75, weights="q4_k_m"),
        # a long prompt the same way
        _case("prompt_block_2048", "prompt_block", "qwen3_4b", 2, 0, 2048, weights="q4_k_m"),
    ]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    op = rng.choice(["decode", "decode", "prefill", "prefill", "token_block", "prompt_block"])
    if op == "decode":
        model = rng.choice(list(MODELS))
        ctx = _log_int(rng, 1, 131072)
        kvd = MODELS[model][1] * MODELS[model][2]
        layers = max(1, min(rng.randint(4, 24), 500_000_000 // (4 * kvd * ctx)))
        return _case("", op, model, layers, ctx - 1, outliers=rng.random() < 0.3)
    if op == "prefill":
        model = rng.choice(list(MODELS))
        n = _log_int(rng, 2, 2048)
        start = 0 if rng.random() < 0.5 else _log_int(rng, 1, 32768)
        nh, hd = MODELS[model][0], MODELS[model][2]
        most = 5e10 if hd in (64, 128) else 5e9
        while 4 * nh * hd * n * (start + n / 2) > most:
            n, start = max(2, n * 2 // 3), start * 2 // 3
        return _case("", op, model, rng.randint(1, 3), start, n)
    if op == "token_block":
        model = rng.choice(["tinyllama", "qwen2.5_0.5b", "qwen3_1.7b", "qwen3_4b", "qwen3_8b", "hd96"])
        weights = "q8_0" if MODELS[model][6] % 512 else rng.choice(["q4_k_m", "q4_k_m", "q8_0", "f16"])
        return _case("", op, model, rng.randint(2, 4), _log_int(rng, 1, 16384) - 1, weights=weights,
                     host=rng.random() < 0.3)
    model = rng.choice(["tinyllama", "qwen2.5_0.5b", "qwen3_1.7b", "qwen3_4b", "qwen3_8b"])
    weights = "q8_0" if MODELS[model][6] % 512 else rng.choice(["q4_k_m", "q4_k_m", "q8_0", "f16"])
    return _case("", op, model, rng.randint(1, 2), 0 if rng.random() < 0.6 else _log_int(rng, 1, 4096),
                 _log_int(rng, 2, 1400), weights=weights, host=rng.random() < 0.2, exact_kv=rng.random() < 0.7)


# ---- inputs, from the seed alone ----

def _seed(seed, what, layer=0):
    return (seed * 1000003 + what * 10007 + layer) & 0x7FFFFFFFFFFF


def _normal(seed, what, layer, shape, dtype=torch.float32):
    g = torch.Generator(device="cuda").manual_seed(_seed(seed, what, layer))
    return torch.randn(shape, generator=g, device="cuda", dtype=dtype)


def _history(case, seed, layer, which, kvd):
    """fp16 cache rows [0, pos) of one layer."""
    n = case["pos"]
    rows = _normal(seed, 1 + which, layer, (n, kvd), torch.float16)
    if case["outliers"]:
        g = torch.Generator(device="cuda").manual_seed(_seed(seed, 3 + which, layer))
        rows *= torch.where(torch.rand(n, 1, generator=g, device="cuda") < 0.01, 8.0, 1.0).half()
    return rows


def _rope_tables(base, hd, n):
    i = np.arange(hd // 2, dtype=np.float32)
    freq = np.power(np.float32(base), 2 * i / np.float32(hd), dtype=np.float32)
    theta = np.arange(n, dtype=np.float32)[:, None] / freq[None, :]
    return np.cos(theta), np.sin(theta)


def _norm_weights(seed, layer, hd):
    r = np.random.RandomState(_seed(seed, 5, layer) & 0x7FFFFFFF)
    return [(1.0 + 0.02 * r.standard_normal(hd)).astype(np.float32) for _ in range(2)]


# the weight types of a file: attn_q, attn_k, attn_v, attn_output
FILES = {"q4_k_m": (Q4_K, Q4_K, Q6_K, Q4_K), "q8_0": (Q8_0,) * 4, "f16": (F16,) * 4}
BLOCK = {F16: (1, 2), Q8_0: (32, 34), Q4_K: (256, 144), Q6_K: (256, 210)}


def _rows(seed, layer, which, wtype, rows, n):
    """GGUF rows as bytes [rows][row bytes], weights of about 1 / sqrt(n)."""
    rng = np.random.default_rng(_seed(seed, 20 + which, layer))
    s = 1.0 / math.sqrt(n)
    if wtype == F16:
        return (rng.standard_normal((rows, n), dtype=np.float32) * np.float32(s)).astype("<f2").view(np.uint8)
    elems, size = BLOCK[wtype]
    nb = n // elems
    raw = rng.integers(0, 256, (rows, nb, size), dtype=np.uint8)

    def put(off, v):
        raw[:, :, off:off + 2] = v.astype("<f2").view(np.uint8).reshape(rows, nb, 2)
    u = rng.uniform(0.5, 1.5, (rows, nb))
    if wtype == Q8_0:
        put(0, u * s / 74)
    elif wtype == Q4_K:
        put(0, u * s / 330)
        put(2, u * s / 44)
    else:
        put(208, u * s / 1360)
    return raw.reshape(rows, nb * size)


def _bias(seed, layer, which, rows):
    rng = np.random.default_rng(_seed(seed, 30 + which, layer))
    return (0.1 * rng.standard_normal(rows)).astype(np.float32)


class _Cache:
    """A context's K or V cache as an array torch can wrap; a tensor made of it keeps the context."""

    def __init__(self, att, ptr, shape):
        self.att = att
        self.__cuda_array_interface__ = {"data": (ptr, False), "shape": shape, "typestr": "<i2", "version": 3}


class _State:
    pass


def prepare(case, seed):
    nh, nkv, hd, rope, base, norm, embd, bias = MODELS[case["model"]]
    L, pos, n = case["layers"], case["pos"], case["n_tok"]
    smax = pos + n
    qd, kvd = nh * hd, nkv * hd
    s = _State()
    s.case = case
    cos, sin = _rope_tables(base, hd, smax)
    s.att = att = PicoAttention(L, smax, nh, nkv, hd, rope, rope_cos=cos, rope_sin=sin)
    s.ext = torch.cuda.ExternalStream(att.stream)
    ptrs = att.kv_cache_ptrs()
    s.kv = [torch.as_tensor(_Cache(att, p, (L, smax, kvd)), device="cuda") for p in ptrs]
    s.new_rows = [c[:, pos:] for c in s.kv]
    if not case["exact_kv"]:  # K and V off the split GEMM: fp16 numbers, not fixed bits
        s.new_rows = [c.view(torch.float16) for c in s.new_rows]
    for l in range(L):
        if norm:
            att.set_qk_norm(l, *_norm_weights(seed, l, hd))
        for i in range(2):
            if pos:
                s.kv[i][l, :pos].copy_(_history(case, seed, l, i, kvd).view(torch.int16))
    if case["weights"]:
        types = FILES[case["weights"]]
        for l in range(L):
            w = [_rows(seed, l, i, types[i], r, embd) for i, r in enumerate((qd, kvd, kvd))]
            b = [_bias(seed, l, i, r) if bias else None for i, r in enumerate((qd, kvd, kvd))]
            bt = F32 if bias else 0
            att.set_qkv_weights(l, embd, w[0], types[0], w[1], types[1], w[2], types[2], b[0], bt, b[1], bt, b[2], bt)
            att.set_out_weights(l, embd, _rows(seed, l, 3, types[3], embd, qd), types[3])
        if not case["exact_kv"]:
            att.set_batch_projection(False)
        s.xb = [_normal(seed, 10, l, (n, embd)) for l in range(L)]
        s.x0 = 0.02 * _normal(seed, 11, 0, (n, embd))  # an embedding row
        s.x = torch.empty_like(s.x0)
        if case["host"]:
            s.xb = [x.cpu().numpy() for x in s.xb]
            s.x0, s.x = s.x0.cpu().numpy(), np.empty((n, embd), np.float32)
    else:
        s.q = [_normal(seed, 12, l, (n, qd)) for l in range(L)]
        s.k = [_normal(seed, 13, l, (n, kvd)) for l in range(L)]
        s.v = [_normal(seed, 14, l, (n, kvd)) for l in range(L)]
        s.out = torch.empty((L, n, qd), device="cuda")
        s.args = [[C.c_void_p(t.data_ptr()) for t in (s.q[l], s.k[l], s.v[l], s.out[l])] for l in range(L)]
    s.graph = None
    if case["graph"]:
        def step():
            for l in range(L):
                check(lib().pqa_decode_noalloc(att.handle, l, pos, *s.args[l]), att.handle)
        torch.cuda.synchronize()
        s.graph = Graph(att.stream, step)
    return s


@contextlib.contextmanager
def _on(s):
    """The context's stream behind torch's current one, and the other way round after the pass."""
    cur = torch.cuda.current_stream()
    s.ext.wait_stream(cur)
    with torch.cuda.stream(s.ext):
        yield
    cur.wait_stream(s.ext)


def run(state):
    s, case = state, state.case
    att, pos, n, L = s.att, case["pos"], case["n_tok"], case["layers"]
    h, op = att.handle, case["op"]
    if s.graph is not None:
        s.graph.launch(torch.cuda.current_stream().cuda_stream)
        return [s.out] + s.new_rows
    if op == "decode":
        f = lib().pqa_decode
        with _on(s):
            for l in range(L):
                check(f(h, l, pos, *s.args[l]), h)
        return [s.out] + s.new_rows
    if op == "prefill":
        f = lib().pqa_prefill
        with _on(s):
            for l in range(L):
                check(f(h, l, pos, n, *s.args[l]), h)
        return [s.out] + s.new_rows
    if case["host"]:
        s.x[:] = s.x0
        for l in range(L):
            if op == "token_block":
                att.attention_block(l, pos, s.xb[l], s.x)
            else:
                att.prefill_block(l, pos, s.xb[l], s.x)
        return [s.x] + s.new_rows
    with _on(s):
        s.x.copy_(s.x0)
        x = C.c_void_p(s.x.data_ptr())
        for l in range(L):
            xb = C.c_void_p(s.xb[l].data_ptr())
            if op == "token_block":
                check(lib().pqa_attention_block(h, l, pos, xb, x), h)
            else:
                check(lib().pqa_prefill_block(h, l, pos, n, xb, x), h)
    return [s.x] + s.new_rows


def work(case):
    nh, nkv, hd, _, _, _, embd, _ = MODELS[case["model"]]
    L, pos, n = case["layers"], case["pos"], case["n_tok"]
    qd, kvd = nh * hd, nkv * hd
    keys = n * pos + n * (n + 1) // 2  # (token, key) pairs of the causal attention
    flops = 4 * qd * keys
    b = 4 * kvd * pos + 4 * kvd * n  # the history read, the new rows written (K and V, fp16)
    if case["weights"]:
        rows = (qd, kvd, kvd)
        for t, r, w in zip(FILES[case["weights"]], rows + (embd,), (embd,) * 3 + (qd,)):
            elems, size = BLOCK[t]
            b += r * (w // elems) * size
            flops += 2 * n * r * w
        b += 4 * n * embd * 3  # xb and x read, x written
    else:
        b += 4 * n * (2 * qd + 2 * kvd)
    return {"bytes": L * b, "flops": L * flops}


def tolerance(case):
    """About four times the largest difference from exact() measured over the kind of case; the appended K and V
    rows are bytes and the same."""
    _, nkv, hd, _, _, _, _, _ = MODELS[case["model"]]
    if case["n_tok"] > 1:
        # head sizes 64 and 128: P in fp16 (2e-4 measured). Others: fp32 throughout; what is left is fp16 rounding
        # of new K rows at near-ties (8e-6)
        return {"rel": 8e-4} if hd in (64, 128) else {"rel": 4e-5}
    if hd in (64, 128) and case["pos"] < 8192 // nkv:
        return {"rel": 6e-4}  # short histories: P in fp16 (1.5e-4)
    return {"rel": 8e-6}  # long ones and other head sizes: fp32 (up to 2e-6)


# ---- the same in 64 bits ----

def _half(b, off):
    return np.ascontiguousarray(b[:, :, off:off + 2]).view("<f2")[..., 0].astype(np.float64)


def _dequant(raw, wtype, n):
    rows = raw.shape[0]
    if wtype == F16:
        w = raw.view("<f2").astype(np.float64)
    else:
        elems, size = BLOCK[wtype]
        b = raw.reshape(rows, n // elems, size)
        if wtype == Q8_0:
            w = _half(b, 0)[..., None] * b[:, :, 2:].view(np.int8)
        elif wtype == Q4_K:  # 8 groups of 32: d sc q - dmin mn, sc and mn in 6 bits
            s = b[:, :, 4:16].astype(np.int32)
            sc = np.concatenate([s[..., 0:4] & 63, (s[..., 8:12] & 15) | ((s[..., 0:4] >> 6) << 4)], -1)
            mn = np.concatenate([s[..., 4:8] & 63, (s[..., 8:12] >> 4) | ((s[..., 4:8] >> 6) << 4)], -1)
            q = b[:, :, 16:].reshape(rows, -1, 4, 32)
            q = np.stack([q & 15, q >> 4], 3).reshape(rows, -1, 8, 32)
            w = (_half(b, 0)[..., None] * sc)[..., None] * q - (_half(b, 2)[..., None] * mn)[..., None]
        else:  # Q6_K: 16 groups of 16 with an int8 scale; 4 low bits and 2 high bits per value
            lo = b[:, :, :128].reshape(rows, -1, 2, 2, 32)
            hi = b[:, :, 128:192].reshape(rows, -1, 2, 32)
            q = np.stack([(lo[:, :, :, g & 1] >> (4 * (g >> 1)) & 15) | ((hi >> (2 * g) & 3) << 4) for g in range(4)], 3)
            sc = b[:, :, 192:208].view(np.int8).reshape(rows, -1, 2, 4, 2, 1)
            w = _half(b, 208)[..., None, None, None, None] * sc * (q.reshape(rows, -1, 2, 4, 2, 16).astype(np.int32) - 32)
    return torch.from_numpy(np.ascontiguousarray(w).reshape(rows, n)).cuda()


def _rope64(x, rope, cos, sin):
    """x [n][heads][hd] rotated; cos and sin [n][hd / 2]."""
    n, heads, hd = x.shape
    if rope == NEOX:
        e0 = torch.arange(hd // 2, device="cuda")
        e1 = e0 + hd // 2
    else:  # blocks of 8: element j of the first four with element j of the last four
        p = torch.arange(hd // 2, device="cuda")
        e0 = (p // 4) * 8 + p % 4
        e1 = e0 + 4
    a, b = x[..., e0], x[..., e1]
    c, d = cos[:, None, :], sin[:, None, :]
    y = torch.empty_like(x)
    y[..., e0], y[..., e1] = a * c - b * d, a * d + b * c
    return y


def _rms64(x, w):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-6) * torch.from_numpy(w).cuda().double()


def _attention64(case, seed, layer, q, k, v, cos, sin):
    """q, k, v in 64 bits [n][heads * hd] -> the block's output [n][q_dim]."""
    nh, nkv, hd, rope, _, norm, _, _ = MODELS[case["model"]]
    n, pos, g = case["n_tok"], case["pos"], nh // nkv
    q, k, v = q.view(n, nh, hd), k.view(n, nkv, hd), v.view(n, nkv, hd)
    if norm:
        qw, kw = _norm_weights(seed, layer, hd)
        q, k = _rms64(q, qw), _rms64(k, kw)
    q, k = _rope64(q, rope, cos, sin), _rope64(k, rope, cos, sin)
    kvd = nkv * hd
    rows = [torch.cat([_history(case, seed, layer, i, kvd).view(pos, nkv, hd), new.half()]) for i, new in ((0, k), (1, v))]
    out = torch.empty((n, nh, hd), dtype=torch.float64, device="cuda")
    later = torch.arange(pos + n, device="cuda")[None, :] > pos + torch.arange(n, device="cuda")[:, None]
    for j in range(nkv):
        kj, vj = rows[0][:, j].double(), rows[1][:, j].double()
        for h in range(j * g, j * g + g):
            sc = q[:, h].contiguous() @ kj.t().contiguous() / math.sqrt(hd)
            out[:, h] = torch.softmax(sc.masked_fill(later, -math.inf), -1) @ vj
    return out.view(n, nh * hd)


def exact(case, seed):
    nh, nkv, hd, rope, base, _, embd, bias = MODELS[case["model"]]
    L, pos, n = case["layers"], case["pos"], case["n_tok"]
    qd, kvd = nh * hd, nkv * hd
    cos, sin = (torch.from_numpy(t[pos:]).cuda().double() for t in _rope_tables(base, hd, pos + n))
    if not case["weights"]:
        outs = []
        for l in range(L):
            q, k, v = (_normal(seed, 12 + i, l, (n, d)).double() for i, d in enumerate((qd, kvd, kvd)))
            outs.append(_attention64(case, seed, l, q, k, v, cos, sin))
        return [torch.stack(outs), None, None]
    types = FILES[case["weights"]]
    x = (0.02 * _normal(seed, 11, 0, (n, embd))).double()
    for l in range(L):
        xb = _normal(seed, 10, l, (n, embd)).double()
        qkv = []
        for i, r in enumerate((qd, kvd, kvd)):
            y = xb @ _dequant(_rows(seed, l, i, types[i], r, embd), types[i], embd).t().contiguous()
            qkv.append(y + torch.from_numpy(_bias(seed, l, i, r)).cuda().double() if bias else y)
        o = _attention64(case, seed, l, *qkv, cos, sin)
        x = x + o @ _dequant(_rows(seed, l, 3, types[3], embd, qd), types[3], qd).t().contiguous()
    return [x, None, None]
