"""Kernels at the edges of their tiles and dispatch ranges, each against the CPU
oracle: partial tiles and stages, the smallest and odd sizes, both sides of each
rule that picks a kernel."""
import numpy as np
import pytest

import oracle as O
from gpu_util import assert_bits_equal
from proj_cases import GEMM_CASES, make_bias, make_rows

torch = pytest.importorskip("torch")
from picolm_qwen_amd import PicoAttention  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _bits(a):
    return np.ascontiguousarray(a, np.float32).view(np.uint32)


# tokens around the 32-wide tile, 36 rows (a partial row tile), widths of less than one
# stage (64 elements; Q8_0 rounds of 256), of a partial last one and of several; K and V of
# different orders in one layer
@pytest.mark.parametrize("n_tok", [1, 31, 32, 33])
@pytest.mark.parametrize("kt,vt,dim", [(O.GGUF_F32, O.GGUF_F16, 8), (O.GGUF_F16, O.GGUF_F32, 200),
                                       (O.GGUF_Q8_0, O.GGUF_Q8_0, 64), (O.GGUF_Q8_0, O.GGUF_Q8_0, 832),
                                       (O.GGUF_Q8_0, O.GGUF_Q6_K, 512), (O.GGUF_Q4_K, O.GGUF_Q8_0, 768)])
def test_ordered_projection_tile_edges(n_tok, kt, vt, dim):
    print(f"reference-order K/V, {n_tok} tokens, types {kt}/{vt}, width {dim}", flush=True)
    rng = np.random.default_rng(100 * dim + n_tok)
    nh, nkv, hd = 4, 2, 18
    att = PicoAttention(1, 64, nh, nkv, hd)
    rows = (nh * hd, nkv * hd, nkv * hd)
    types = (kt, kt, vt)
    w = [make_rows(rng, t, r, dim) for t, r in zip(types, rows)]
    bt = (O.GGUF_NONE, O.GGUF_F32, O.GGUF_F16)
    b = [None, make_bias(rng, bt[1], rows[1]), make_bias(rng, bt[2], rows[2])]
    att.set_qkv_weights(0, dim, w[0], types[0], w[1], types[1], w[2], types[2], b[0], bt[0], b[1], bt[1], b[2], bt[2])
    x = rng.standard_normal((n_tok, dim)).astype(np.float32)
    _, k, v = (g.cpu().numpy() for g in att.qkv_project_batch(0, torch.from_numpy(x).to(DEV)))
    for name, g, j in (("k", k, 1), ("v", v, 2)):
        assert_bits_equal(_bits(g), _bits(O.matmul_bias_tokens(x, w[j], types[j], rows[j], b[j], bt[j])), name)
    att.close()


# infinities, NaN, subnormals, zeros of both signs and products that overflow or vanish, in weights and
# inputs: every K and V element is the oracle's bits, or NaN where its is NaN
@pytest.mark.parametrize("n_tok", [3, 300])  # 16 x 16 and 32 x 32 tiles
@pytest.mark.parametrize("kt", [O.GGUF_F32, O.GGUF_F16, O.GGUF_Q8_0])
def test_ordered_projection_special_values(kt, n_tok):
    print(f"reference-order K/V of special values, type {kt}, {n_tok} tokens", flush=True)
    rng = np.random.default_rng(900 + kt + n_tok)
    nkv, hd, dim = 8, 128, 320
    att = PicoAttention(1, 16, nkv, nkv, hd)
    rows = nkv * hd
    w = [make_rows(rng, kt, rows, dim, special=True) for _ in range(3)]
    special = np.array([np.inf, -np.inf, np.nan, 0.0, -0.0, 1e-45, -1e-40, 1.2e-38, 3e38, -3e38, 2e-23], np.float32)
    x = rng.standard_normal((n_tok, dim)).astype(np.float32)
    x[rng.random(x.shape) < 0.3] *= np.float32(1e-38)
    at = rng.random(x.shape) < 0.3
    x[at] = rng.choice(special[3:], at.sum()) / (1 if kt == O.GGUF_F32 else 2048)  # int8 and fp16 weights are larger
    for t in range(0, n_tok, 3):  # a third of the tokens, so that most sums stay finite
        x[t, 11], x[t, 200] = np.inf, special[t // 3 % 3]
    x[-1] = rng.standard_normal(dim)
    for m in w:
        if kt == O.GGUF_Q8_0:
            m.reshape(rows, dim // 32, 34)[::7, 3, :2] = np.array([0x7C00], "<u2").view(np.uint8)  # infinite scales
            continue
        f = m.view("<f4" if kt == O.GGUF_F32 else "<f2").reshape(rows, dim)
        finite = special[3:] if kt == O.GGUF_F32 else np.array([0.0, -0.0, 6e-8, -3e-6, 6.2e-5, 65504, -65504], np.float32)
        at = rng.random(f.shape) < 0.2
        f[at] = rng.choice(finite, at.sum())
        f[::5, 17] = rng.choice(np.concatenate([special[:3], finite]), rows // 5 + 1)
    att.set_qkv_weights(0, dim, w[0], kt, w[1], kt, w[2], kt)
    _, k, v = (g.cpu().numpy() for g in att.qkv_project_batch(0, torch.from_numpy(x).to(DEV)))
    for name, g, m in (("k", k, w[1]), ("v", v, w[2])):
        want = O.matmul_bias_tokens(x, m, kt, rows)
        nan = np.isnan(want)
        assert 0.01 < nan.mean() < 0.9 and np.isinf(want).any()
        assert np.array_equal(np.isnan(g), nan), name
        assert_bits_equal(_bits(np.where(nan, 0, g)), _bits(np.where(nan, 0, want)), name)
    att.close()


# the split GEMM's workgroup tiles (64 to 256 rows, 64 to 192 columns, each with and without K
# slices): the shapes of GEMM_CASES, whose plans a CPU test checks
@pytest.mark.parametrize("n_tok,dim,nh,out_rows", [c[:4] for c in GEMM_CASES])
def test_split_gemm_tile_edges(n_tok, dim, nh, out_rows):
    print(f"split GEMM, {n_tok} tokens, width {dim}, {nh} heads, {out_rows} output rows", flush=True)
    assert torch.cuda.get_device_properties(0).multi_processor_count == 256  # what the plans are for
    rng = np.random.default_rng(7 * n_tok + dim)
    nkv, hd, wt = 1, 64, O.GGUF_F32
    att = PicoAttention(1, 16, nh, nkv, hd)
    rows = (nh * hd, hd, hd)
    w = [make_rows(rng, wt, r, dim) for r in rows]
    b = make_bias(rng, O.GGUF_F32, rows[0])
    att.set_qkv_weights(0, dim, w[0], wt, w[1], wt, w[2], wt, b, O.GGUF_F32)
    wo, bo = make_rows(rng, wt, out_rows, nh * hd), make_bias(rng, O.GGUF_F32, out_rows)
    att.set_out_weights(0, out_rows, wo, wt, bo, O.GGUF_F32)
    wf = [m.view(np.float32).astype(np.float64) for m in (*w, wo)]
    # every token of a small prompt, the edges of every tile and some within of a large one
    some = np.arange(n_tok) if n_tok * dim * nh < 1e8 else np.array(
        sorted({0, 1, n_tok - 1} | {t + d for t in range(64, n_tok, 64) for d in (-1, 0)} | set(range(5, n_tok, 97))))

    def check(got, x, wm, bias, residual, name):
        x = x[some].astype(np.float64)
        want = x @ wm.T + bias
        mag = np.abs(x) @ np.abs(wm).T
        got = got[some].astype(np.float64)
        # 3 n products of 22-bit operands: within (3 n + 12) 2^-24 sum |w x| of the exact sum, and a rounding of the
        # bias sum (and of the residual sum) on top
        last = 2.0 ** -23 * (np.abs(want) + (np.abs(want + residual) if residual is not None else 0))
        full = want if residual is None else want + residual
        err = np.abs(got - full)
        assert np.all(err <= (3 * wm.shape[1] + 12) * 2.0 ** -24 * mag + last + 1e-30), name
        # and in the mean square (less that last rounding) far below what a product without a low part would be off,
        # 2^-12.2 of sqrt(sum w^2 x^2): the split gives 2^-23.7 of it, the fp32 sums at most 2^-24 sqrt(3 n)
        rms = np.sqrt(np.mean(np.maximum(err - last, 0) ** 2))
        assert rms <= 2.0 ** -17 * np.sqrt(np.mean((x * x) @ (wm * wm).T)), (name, rms)

    x = rng.standard_normal((n_tok, dim)).astype(np.float32)
    for exact_kv in (False, True):
        att.set_batch_projection(exact_kv)
        got = [g.cpu().numpy() for g in att.qkv_project_batch(0, torch.from_numpy(x).to(DEV))]
        for j in range(1 if exact_kv else 3):
            check(got[j], x, wf[j], b.view(np.float32) if j == 0 else 0.0, None, "qkv"[j])
    a = rng.standard_normal((n_tok, nh * hd)).astype(np.float32)
    x0 = rng.standard_normal((n_tok, out_rows)).astype(np.float32)
    xo = torch.from_numpy(x0.copy()).to(DEV)
    att.out_project_batch(0, torch.from_numpy(a).to(DEV), xo)
    check(xo.cpu().numpy(), a, wf[3], bo.view(np.float32), x0[some], "out")
    att.close()


# prefill behind a history: blocks whose keys are cut into ranges (few blocks, a long history),
# ranges past a row's own position and empty ones of the first blocks (a prompt at 0), one block
# per workgroup without ranges, and prompts that stay on block pairs; both head sizes, both q precisions
@pytest.mark.parametrize("nh,nkv,hd,start,n_tok,split_q", [(4, 1, 64, 3000, 5, True), (2, 1, 128, 1000, 100, True),
                                                           (7, 1, 64, 700, 65, False), (8, 2, 128, 2047, 1, True),
                                                           (4, 2, 128, 64, 300, True), (32, 2, 64, 129, 700, True),
                                                           (32, 1, 128, 500, 2100, False),
                                                           (2, 1, 128, 0, 2048, True), (8, 2, 128, 3000, 40, False),
                                                           (4, 1, 64, 0, 1500, False)])
def test_prefill_key_ranges(nh, nkv, hd, start, n_tok, split_q):
    print(f"prefill ranges {nh}/{nkv} x {hd}, {n_tok} tokens at {start}, split_q {split_q}", flush=True)
    smax, seed, kvd = start + n_tok, 4100 + start, nkv * hd
    cos, sin = O.rope_table(1e6, hd, smax)
    att = PicoAttention(1, smax, nh, nkv, hd, 0, rope_cos=cos, rope_sin=sin)
    att.set_prefill_precision(split_q)
    att.synth_kv(0, 0, start, seed, 0.0)
    kc, vc = np.zeros((smax, kvd), np.uint16), np.zeros((smax, kvd), np.uint16)
    kc[:start], vc[:start] = O.synth_kv_rows(seed, 0, kvd, 0, start, 0.0)
    q, k, v = O.batch_inputs(seed, 0, 0, n_tok, nh, nkv, hd)
    out = att.forward_batch(0, start, *(torch.from_numpy(x).to(DEV) for x in (q, k, v))).cpu().numpy()
    shp = O.shape(nh, nkv, hd, smax, 0)
    qr = [O.append(shp, start + t, q[t], k[t], v[t], None, None, cos[start + t], sin[start + t], kc, vc)
          for t in range(n_tok)]
    gk, gv = att.kv_download(0, start, n_tok)
    assert_bits_equal(gk, kc[start:], "K rows")
    assert_bits_equal(gv, vc[start:], "V rows")
    # P is rounded to fp16 for the PV product and its own sum (2^-11 each, relative to sum p |v|); one fp16 q
    # moves a score by up to 2^-11 |q| |k| / sqrt(hd) (log2 units included), about 2^-8 at these N(0, 1) rows
    rel = 2.0 ** -10 if split_q else 2.0 ** -6
    for t in sorted({0, 1, n_tok // 2, n_tok - 2, n_tok - 1} & set(range(n_tok))):
        want = O.attend_f64(shp, start + t, qr[t], kc, vc)
        mag = O.attend_f64(shp, start + t, qr[t], kc, vc & 0x7FFF)
        assert np.all(np.abs(out[t] - want) <= rel * mag + 1e-6), t
    att.close()


# the matrix-core kernels of the other head sizes: history lengths around their 32-key tiles, one
# and several tiles per wave, one and several key ranges (decode and prefill), GQA groups of 1 to
# 20 heads (more than 16: two row blocks), every size and RoPE pairing
GEN = [(80, 4, 4, 0), (96, 8, 2, 31), (112, 7, 1, 32), (160, 20, 1, 33), (192, 6, 2, 127), (256, 8, 1, 128),
       (80, 17, 1, 513), (96, 32, 8, 3001), (256, 16, 2, 2500), (160, 3, 3, 1100), (112, 12, 4, 4100), (192, 2, 1, 700)]


def _gen_case(hd, nh, nkv, start, n_tok, style, seed):
    smax, kvd = start + n_tok, nkv * hd
    cos, sin = O.rope_table(1e6, hd, smax)
    att = PicoAttention(1, smax, nh, nkv, hd, style, rope_cos=cos, rope_sin=sin)
    qn, kn = O.qk_norm_weights(seed, 0, hd)
    att.set_qk_norm(0, qn, kn)
    att.synth_kv(0, 0, start, seed, 0.01)
    kc, vc = np.zeros((smax, kvd), np.uint16), np.zeros((smax, kvd), np.uint16)
    kc[:start], vc[:start] = O.synth_kv_rows(seed, 0, kvd, 0, start, 0.01)
    q, k, v = O.batch_inputs(seed, 0, 0, n_tok, nh, nkv, hd)
    return att, q, k, v, qn, kn, cos, sin, kc, vc


def _check_gen(att, shp, start, toks, out, q, k, v, qn, kn, cos, sin, kc, vc):
    qr = [O.append(shp, start + t, q[t], k[t], v[t], qn, kn, cos[start + t], sin[start + t], kc, vc)
          for t in range(q.shape[0])]
    gk, gv = att.kv_download(0, start, q.shape[0])
    assert_bits_equal(gk, kc[start:], "K rows")
    assert_bits_equal(gv, vc[start:], "V rows")
    for t in toks:
        want = O.attend_f64(shp, start + t, qr[t], kc, vc)
        mag = O.attend_f64(shp, start + t, qr[t], kc, vc & 0x7FFF)
        # 22-bit operands and fp32 sums: a score is off by at most 2^-20 sum |q k| log2(e) / sqrt(hd), with the x8
        # outlier rows below 2^-20 * 150; twice that, times ln 2, relative to sum p |v|
        assert np.all(np.abs(out[t] - want) <= 2.0 ** -12 * mag), t
        # and in the mean square far below it
        assert np.sqrt(np.mean((out[t] - want) ** 2)) <= 2.0 ** -18 * np.sqrt(np.mean(mag ** 2)), t


@pytest.mark.parametrize("hd,nh,nkv,pos", GEN)
def test_general_mma_decode(hd, nh, nkv, pos):
    style, seed = (hd // 16) % 3, 5100 + pos
    print(f"general decode {nh}/{nkv} x {hd} at {pos}, rope {style}", flush=True)
    att, q, k, v, qn, kn, cos, sin, kc, vc = _gen_case(hd, nh, nkv, pos, 1, style, seed)
    out = att.forward(0, pos, *(torch.from_numpy(x[0]).to(DEV) for x in (q, k, v))).cpu().numpy()
    _check_gen(att, O.shape(nh, nkv, hd, pos + 1, style), pos, [0], out[None], q, k, v, qn, kn, cos, sin, kc, vc)
    att.close()


@pytest.mark.parametrize("n_tok", [1, 17, 70])
@pytest.mark.parametrize("hd,nh,nkv,start", GEN)
def test_general_mma_prefill(hd, nh, nkv, start, n_tok):
    style, seed = (hd // 16 + 1) % 3, 5200 + start
    print(f"general prefill {nh}/{nkv} x {hd}, {n_tok} tokens at {start}, rope {style}", flush=True)
    att, q, k, v, qn, kn, cos, sin, kc, vc = _gen_case(hd, nh, nkv, start, n_tok, style, seed)
    flat = torch.empty(n_tok * nh * hd + 2, device=DEV)
    o = flat[2:].view(n_tok, nh * hd)  # 8-byte aligned output, 4-byte aligned q
    qd = torch.empty(q.size + 1, device=DEV)[1:].view(q.shape)
    qd.copy_(torch.from_numpy(q))
    att.forward_batch(0, start, qd, torch.from_numpy(k).to(DEV), torch.from_numpy(v).to(DEV), out=o)
    out = o.cpu().numpy()
    _check_gen(att, O.shape(nh, nkv, hd, start + n_tok, style), start, sorted({0, n_tok // 2, n_tok - 1}), out, q, k, v,
               qn, kn, cos, sin, kc, vc)
    att.close()


@pytest.mark.parametrize("hd", [80, 96, 256])
def test_general_mma_non_finite_rows(hd):
    # rows that overflow fp16 (infinities in the cache): tokens before them are untouched, a key of score -inf
    # has weight 0, and what is infinite or NaN in the reference's arithmetic stays so
    print(f"general path, infinite cache rows, hd {hd}", flush=True)
    nh, nkv, n_tok, seed = 4, 1, 45, 5300 + hd
    cos, sin = np.ones((n_tok, hd // 2), np.float32), np.zeros((n_tok, hd // 2), np.float32)  # no rotation
    att = PicoAttention(1, n_tok, nh, nkv, hd, 0, rope_cos=cos, rope_sin=sin)
    q, k, v = (x.copy() for x in O.batch_inputs(seed, 0, 0, n_tok, nh, nkv, hd))
    q[:, 0::hd] = np.abs(q[:, 0::hd]) + 0.1   # dim 0 of every head: positive, and
    k[20, 0] = -1e6                           # row 20's score -inf
    v[33, 5] = 1e6                            # dim 5 infinite from token 33 on
    v[40, 7] = np.nan
    out = att.forward_batch(0, 0, *(torch.from_numpy(x).to(DEV) for x in (q, k, v))).cpu().numpy()
    shp = O.shape(nh, nkv, hd, n_tok, 0)
    kc, vc = np.zeros((n_tok, nkv * hd), np.uint16), np.zeros((n_tok, nkv * hd), np.uint16)
    for t in range(n_tok):
        qr = O.append(shp, t, q[t], k[t], v[t], None, None, cos[t], sin[t], kc, vc)
        want = O.attend(shp, t, qr, kc, vc)
        assert np.array_equal(np.isnan(out[t]), np.isnan(want)), t
        assert np.array_equal(np.isinf(out[t]), np.isinf(want)), t
        fin = np.isfinite(want)
        assert np.all(np.abs(out[t][fin] - want[fin]) <= 1e-4), t
    # the same through the decode: the last token again, over the rows just written
    t = n_tok - 1
    dec = att.forward(0, t, *(torch.from_numpy(x[t]).to(DEV) for x in (q, k, v))).cpu().numpy()
    assert np.array_equal(np.isnan(dec), np.isnan(want)) and np.array_equal(np.isinf(dec), np.isinf(want))
    att.close()


# prompts with enough 32 x 32 tiles for two waves per SIMD (the smaller ones above run 16 x 16)
@pytest.mark.parametrize("kt,vt,dim", [(O.GGUF_Q8_0, O.GGUF_Q8_0, 320), (O.GGUF_F16, O.GGUF_F16, 136)])
def test_ordered_projection_many_tiles(kt, vt, dim):
    print(f"reference-order K/V, 270 tokens x 2 x 1024 rows, types {kt}/{vt}, width {dim}", flush=True)
    rng = np.random.default_rng(dim)
    nkv, hd, n_tok = 8, 128, 270
    att = PicoAttention(1, 16, nkv, nkv, hd)
    rows = nkv * hd
    w = [make_rows(rng, t, rows, dim) for t in (kt, kt, vt)]
    att.set_qkv_weights(0, dim, w[0], kt, w[1], kt, w[2], vt)
    x = rng.standard_normal((n_tok, dim)).astype(np.float32)
    _, k, v = (g.cpu().numpy() for g in att.qkv_project_batch(0, torch.from_numpy(x).to(DEV)))
    assert_bits_equal(_bits(k), _bits(O.matmul_bias_tokens(x, w[1], kt, rows)), "k")
    assert_bits_equal(_bits(v), _bits(O.matmul_bias_tokens(x, w[2], vt, rows)), "v")
    att.close()


# the same through the host entries, whose decode reads q, k and v and writes out in pinned host memory
@pytest.mark.parametrize("hd", [80, 256])
def test_general_mma_host_decode(hd):
    print(f"general decode from host memory, hd {hd}", flush=True)
    nh, nkv, pos, seed = 6, 2, 700, 5400 + hd
    att, q, k, v, qn, kn, cos, sin, kc, vc = _gen_case(hd, nh, nkv, pos, 1, 0, seed)
    dev = att.forward(0, pos, *(torch.from_numpy(x[0]).to(DEV) for x in (q, k, v))).cpu().numpy()
    out = np.asarray(att.forward(0, pos, q[0], k[0], v[0]))
    assert_bits_equal(_bits(out), _bits(dev), "host against device entry")
    _check_gen(att, O.shape(nh, nkv, hd, pos + 1, 0), pos, [0], out[None], q, k, v, qn, kn, cos, sin, kc, vc)
    att.close()


# many small weights beside one large one (an attention sink with a small V row): what the other keys add is
# then the whole output, at weights of 2^-31 to 2^-24 or 2^-30 of the largest; matrix-core sizes and VALU ones (72, 100)
@pytest.mark.parametrize("span", [7.0, 1.0])
@pytest.mark.parametrize("n_tok", [0, 20])  # 0: a decode
@pytest.mark.parametrize("hd", [72, 80, 96, 100, 112, 160, 192, 256])
def test_general_small_weights_beside_a_sink(hd, n_tok, span):
    print(f"general path, weights 2^-31 to 2^-{31 - span:g} beside a sink, hd {hd}, {n_tok} tokens", flush=True)
    rng = np.random.default_rng(5500 + hd)
    nh, nkv, start, n = 4, 1, 3000, max(1, n_tok)
    smax = start + n
    cos, sin = np.ones((smax, hd // 2), np.float32), np.zeros((smax, hd // 2), np.float32)  # no rotation
    att = PicoAttention(1, smax, nh, nkv, hd, 0, rope_cos=cos, rope_sin=sin)
    unit = np.sqrt(hd) / 1.4426950408889634  # a product of q and k that is one log2 unit of score
    k = np.zeros((smax, hd), np.float32)
    k[:, 1] = rng.uniform(0, span, smax) * unit
    k[0, 0], k[0, 1] = 31 * unit / 8, 0
    v = rng.standard_normal((smax, hd)).astype(np.float32)
    v[0] = 0
    q = np.zeros((n, nh, hd), np.float32)
    q[..., 0], q[..., 1] = 8, 1
    q = q.reshape(n, -1)
    kc, vc = (m[:start].astype(np.float16).view(np.uint16) for m in (k, v))
    att.kv_upload(0, 0, kc, vc)
    kc, vc = (np.concatenate([m, np.zeros((n, hd), np.uint16)]) for m in (kc, vc))
    args = [torch.from_numpy(np.ascontiguousarray(x)).to(DEV) for x in (q, k[start:], v[start:])]
    if n_tok:
        out = att.forward_batch(0, start, *args).cpu().numpy()
    else:
        out = att.forward(0, start, *(x[0].contiguous() for x in args)).cpu().numpy()[None]
    shp = O.shape(nh, nkv, hd, smax, 0)
    for t in range(n):
        qr = O.append(shp, start + t, q[t], k[start + t], v[start + t], None, None, cos[0], sin[0], kc, vc)
        want = O.attend_f64(shp, start + t, qr, kc, vc)
        mag = O.attend_f64(shp, start + t, qr, kc, vc & 0x7FFF)
        # a score of 31 log2 units has an fp32 step of 2^-19, q 22 bits: 2^-18 of a weight, and as much again for
        # the weight itself
        err = np.sqrt(np.mean((out[t] - want) ** 2)) / np.sqrt(np.mean(mag ** 2))
        if t in (0, n - 1):
            print(f"  token {t}: {err:.2e} of sum p |v|", flush=True)
        assert err <= 2.0 ** -17, t
    att.close()


# the same rows among several key ranges (decode: several waves and workgroups; prefill: blocks cut in two or
# more), with infinite and NaN rows in the first, a middle and the last range, the new rows among them; groups of
# rows at one position and at sixteen
@pytest.mark.parametrize("hd,nh,nkv", [(80, 4, 4), (96, 8, 2), (112, 17, 1), (160, 4, 1), (192, 2, 2), (256, 8, 2)])
def test_general_mma_non_finite_rows_in_ranges(hd, nh, nkv):
    print(f"general path, infinite cache rows in several ranges, {nh}/{nkv} x {hd}", flush=True)
    start, n_tok, seed, kvd = 2100, 40, 5600 + hd, nkv * hd
    smax = start + n_tok
    cos, sin = np.ones((smax, hd // 2), np.float32), np.zeros((smax, hd // 2), np.float32)  # no rotation
    att = PicoAttention(1, smax, nh, nkv, hd, 0, rope_cos=cos, rope_sin=sin)
    kc, vc = np.zeros((smax, kvd), np.uint16), np.zeros((smax, kvd), np.uint16)
    kc[:start], vc[:start] = O.synth_kv_rows(seed, 0, kvd, 0, start, 0.0)
    inf, ninf = 0x7C00, 0xFC00
    kc[[5, 1000, 2090], 0::hd] = ninf  # dim 0 of q is positive: score -inf, weight 0
    vc[3, 4], vc[3, 9] = inf, 0x7E00   # infinite and NaN in every output
    vc[1111, 6] = ninf
    vc[2095, 8] = inf
    q, k, v = (x.copy() for x in O.batch_inputs(seed, 0, 0, n_tok, nh, nkv, hd))
    q[:, 0::hd] = np.abs(q[:, 0::hd]) + 0.1
    k[7, 0] = -1e6
    v[20, 10] = 1e6   # dim 10 infinite from token 20 on
    v[33, 12] = -1e6  # and a new token whose own row is infinite
    v[33, 6] = 1e6    # +inf after -inf: NaN from token 33 on
    att.kv_upload(0, 0, kc[:start], vc[:start])
    dq, dk, dv = (torch.from_numpy(x).to(DEV) for x in (q, k, v))
    out = att.forward_batch(0, start, dq, dk, dv).cpu().numpy()
    shp = O.shape(nh, nkv, hd, smax, 0)
    dec = {}
    for t in (0, 19, 20, 33, n_tok - 1):  # the decode of a token, over the rows the prompt left before it
        dec[t] = att.forward(0, start + t, dq[t].contiguous(), dk[t].contiguous(), dv[t].contiguous()).cpu().numpy()
    for t in range(n_tok):
        qr = O.append(shp, start + t, q[t], k[t], v[t], None, None, cos[0], sin[0], kc, vc)
        want = O.attend(shp, start + t, qr, kc, vc)
        assert np.isfinite(want).any() and np.isinf(want).any() and np.isnan(want).any()
        for got in [out[t]] + ([dec[t]] if t in dec else []):
            assert np.array_equal(np.isnan(got), np.isnan(want)), t
            assert np.array_equal(got[np.isinf(want)], want[np.isinf(want)]), t
            fin = np.isfinite(want)
            assert np.all(np.abs(got[fin] - want[fin]) <= 1e-4), t
    att.close()
