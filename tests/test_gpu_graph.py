"""pqa_decode_noalloc captured into a HIP graph (picolm_qwen_amd.hipgraph) and
replayed: every replay, with eager work and synchronisations of the program
between replays, gives pqa_decode's outputs bit for bit, for one-launch
per-column steps, split + merge steps and whole-row workgroups; and pqa_prefill
the same way."""
import ctypes as C

import numpy as np
import pytest

import oracle as O

torch = pytest.importorskip("torch")
from picolm_qwen_amd import PicoAttention, _lib  # noqa: E402
from picolm_qwen_amd.hipgraph import Graph  # noqa: E402

pytestmark = pytest.mark.gpu
DEV = torch.device("cuda:0")


def _ptr(t):
    return C.c_void_p(t.data_ptr())


@pytest.mark.parametrize("nh,nkv,hd,pos", [
    (14, 2, 64, 5),        # one split per column, one launch
    (14, 2, 64, 1500),     # per-column splits + the one-wave merge launch
    (16, 8, 128, 8191),    # whole-row workgroups + the merge launch
])
def test_graph_replays_equal_eager_decode(nh, nkv, hd, pos):
    print(f"graph replay {nh}/{nkv}/{hd} pos {pos}", flush=True)
    n_layers, seed = 2, 9100 + pos
    cos, sin = O.rope_table(1e6, hd, pos + 1)
    att = PicoAttention(n_layers, pos + 1, nh, nkv, hd, 0, rope_cos=cos, rope_sin=sin)
    for layer in range(n_layers):
        att.set_qk_norm(layer, *O.qk_norm_weights(seed, layer, hd))
        att.synth_kv(layer, 0, pos, seed + layer, 0.01)
    L = _lib.lib()
    ins = [tuple(torch.from_numpy(x).to(DEV) for x in O.step_inputs(seed, layer, pos, nh, nkv, hd))
           for layer in range(n_layers)]
    want = [torch.zeros(nh * hd, device=DEV) for _ in range(n_layers)]
    got = [torch.zeros(nh * hd, device=DEV) for _ in range(n_layers)]
    torch.cuda.synchronize()
    for layer in range(n_layers):
        q, k, v = ins[layer]
        assert L.pqa_decode(att.handle, layer, pos, _ptr(q), _ptr(k), _ptr(v), _ptr(want[layer])) == 0
    att.sync()
    stream = L.pqa_stream(att.handle)

    def step():
        for layer in range(n_layers):
            q, k, v = ins[layer]
            rc = L.pqa_decode_noalloc(att.handle, layer, pos, _ptr(q), _ptr(k), _ptr(v), _ptr(got[layer]))
            assert rc == 0, att.last_error()

    g = Graph(stream, step)
    x = torch.randn(512, 512, device=DEV)
    for rep in range(4):
        for t in got:
            t.zero_()
        y = x @ x  # the program's own eager work between replays
        torch.cuda.synchronize()
        g.launch(stream)
        att.sync()
        torch.cuda.synchronize()
        for layer in range(n_layers):
            assert torch.equal(got[layer].view(torch.int32), want[layer].view(torch.int32)), (rep, layer)
        assert torch.isfinite(y).all()
    g.close()
    att.close()


def test_graph_replays_equal_eager_prefill():
    # pqa_prefill of two layers (Qwen3-4B heads, a 40-row history) captured
    # and replayed with the new cache rows cleared between replays: every
    # replay rewrites them, and its outputs and rows equal the eager call's
    print("graph replay prefill", flush=True)
    nh, nkv, hd, smax, start, n, seed = 32, 8, 128, 512, 40, 300, 9200
    cos, sin = O.rope_table(1e6, hd, smax)
    att = PicoAttention(2, smax, nh, nkv, hd, 0, rope_cos=cos, rope_sin=sin)
    for layer in range(2):
        att.set_qk_norm(layer, *O.qk_norm_weights(seed, layer, hd))
        att.synth_kv(layer, 0, start, seed + layer, 0.0)
    L = _lib.lib()
    ins = [tuple(torch.from_numpy(x).to(DEV) for x in O.batch_inputs(seed, layer, start, n, nh, nkv, hd))
           for layer in range(2)]
    want = [torch.zeros(n, nh * hd, device=DEV) for _ in range(2)]
    got = [torch.zeros(n, nh * hd, device=DEV) for _ in range(2)]
    torch.cuda.synchronize()
    for layer in range(2):
        q, k, v = ins[layer]
        assert L.pqa_prefill(att.handle, layer, start, n, _ptr(q), _ptr(k), _ptr(v), _ptr(want[layer])) == 0
    att.sync()
    rows = [att.kv_download(layer, start, n) for layer in range(2)]
    zeros = np.zeros((n, nkv * hd), np.uint16)
    stream = L.pqa_stream(att.handle)

    def step():
        for layer in range(2):
            q, k, v = ins[layer]
            rc = L.pqa_prefill(att.handle, layer, start, n, _ptr(q), _ptr(k), _ptr(v), _ptr(got[layer]))
            assert rc == 0, att.last_error()

    g = Graph(stream, step)
    for rep in range(3):
        for layer in range(2):
            got[layer].zero_()
            att.kv_upload(layer, start, zeros, zeros)
        torch.cuda.synchronize()
        g.launch(stream)
        att.sync()
        for layer in range(2):
            assert torch.equal(got[layer].view(torch.int32), want[layer].view(torch.int32)), (rep, layer)
            gk, gv = att.kv_download(layer, start, n)
            assert np.array_equal(gk, rows[layer][0]) and np.array_equal(gv, rows[layer][1]), (rep, layer)
    g.close()
    att.close()


def test_shorter_prompt_after_a_longer_one_needs_no_new_workspace():
    # a warm-up with the longest prompt covers every shorter one, also where the shorter one's GEMMs
    # are cut into K slices and the longer one's are not (137 tokens, 4 slices; 138, one): its capture
    # allocates nothing, and the longer prompt's graph keeps its buffers, in both K/V projection modes
    print("graph prompt blocks, 138 then 137 and 20 tokens", flush=True)
    rng = np.random.default_rng(9300)
    nh, nkv, hd, dim, smax = 32, 8, 128, 2560, 160
    att = PicoAttention(1, smax, nh, nkv, hd, 0)
    w = [(rng.standard_normal((r, n), dtype=np.float32) / np.sqrt(n)).astype(np.float16).view(np.uint8)
         for r, n in ((nh * hd, dim), (nkv * hd, dim), (nkv * hd, dim), (dim, nh * hd))]
    att.set_qkv_weights(0, dim, *(a for m in w[:3] for a in (m, O.GGUF_F16)))
    att.set_out_weights(0, dim, w[3], O.GGUF_F16)
    L = _lib.lib()
    stream = L.pqa_stream(att.handle)
    for exact_kv in (True, False):
        att.set_batch_projection(exact_kv)
        runs = []
        for n in (138, 137, 20):
            xb = torch.from_numpy(rng.standard_normal((n, dim)).astype(np.float32)).to(DEV)
            runs.append([n, xb, torch.zeros(n, dim, device=DEV), None, None])
        torch.cuda.synchronize()

        def block(run):
            assert L.pqa_prefill_block(att.handle, 0, 0, run[0], _ptr(run[1]), _ptr(run[2])) == 0, att.last_error()

        block(runs[0])  # the longest prompt, once
        att.sync()
        for run in runs:
            run[3] = Graph(stream, lambda: block(run))
        for run in runs:
            run[2].zero_()
            torch.cuda.synchronize()
            block(run)
            att.sync()
            run[4] = run[2].clone()
        for rep in range(3):
            for run in runs:
                run[2].zero_()
                torch.cuda.synchronize()
                run[3].launch(stream)
                att.sync()
                assert torch.equal(run[2].view(torch.int32), run[4].view(torch.int32)), (exact_kv, run[0], rep)
        for run in runs:
            run[3].close()
    att.close()


class _KernelNodeParams(C.Structure):  # hipKernelNodeParams
    _fields_ = [("block", C.c_uint32 * 3), ("extra", C.c_void_p), ("func", C.c_void_p), ("grid", C.c_uint32 * 3),
                ("args", C.POINTER(C.c_void_p)), ("shared", C.c_uint32)]


def _last_kernel_first_pointer(g):
    """The first argument of the last kernel of a captured chain: the partials that the merge of key
    ranges reads."""
    hip = C.CDLL("libamdhip64.so.7")
    n = C.c_size_t()
    assert hip.hipGraphGetNodes(g.graph, None, C.byref(n)) == 0
    nodes = (C.c_void_p * n.value)()
    assert hip.hipGraphGetNodes(g.graph, nodes, C.byref(n)) == 0
    last = []
    for node in nodes:
        deg = C.c_size_t()
        assert hip.hipGraphNodeGetDependentNodes(C.c_void_p(node), None, C.byref(deg)) == 0
        if deg.value == 0:
            last.append(node)
    assert len(last) == 1 and n.value == 3, (len(last), n.value)  # K/V rows, attention, merge
    p = _KernelNodeParams()
    assert hip.hipGraphKernelNodeGetParams(C.c_void_p(last[0]), C.byref(p)) == 0
    return C.cast(p.args[0], C.POINTER(C.c_void_p))[0]


@pytest.mark.parametrize("nh,nkv,hd,start,n", [(8, 2, 128, 3000, 40), (8, 2, 64, 3000, 33), (8, 2, 96, 3000, 40)])
def test_captured_prompts_of_two_layers_replayed_at_once(nh, nkv, hd, start, n):
    # prompts whose keys are cut into ranges, captured per layer without an earlier call and replayed on
    # two streams at once, with an eager one of a third layer on the context's stream: each has partials
    # of its own, and every result equals the eager call's
    print(f"graphs at once, {n} tokens at {start}, head size {hd}", flush=True)
    seed = 9400 + hd
    cos, sin = O.rope_table(1e6, hd, start + n)
    att = PicoAttention(3, start + n, nh, nkv, hd, 0, rope_cos=cos, rope_sin=sin)
    L = _lib.lib()
    ins, got = [], [torch.zeros(n, nh * hd, device=DEV) for _ in range(3)]
    for layer in range(3):
        att.synth_kv(layer, 0, start, seed + layer, 0.01)
        ins.append([torch.from_numpy(x).to(DEV) for x in O.batch_inputs(seed, layer, 0, n, nh, nkv, hd)])
    torch.cuda.synchronize()

    def call(layer):
        q, k, v = ins[layer]
        assert L.pqa_prefill(att.handle, layer, start, n, _ptr(q), _ptr(k), _ptr(v), _ptr(got[layer])) == 0, att.last_error()

    stream = L.pqa_stream(att.handle)
    graphs = [Graph(stream, lambda layer=layer: call(layer)) for layer in range(2)]
    parts = [_last_kernel_first_pointer(g) for g in graphs]
    assert parts[0] and parts[1] and parts[0] != parts[1]
    again = Graph(stream, lambda: call(0))  # a layer's later captures use its buffer
    assert _last_kernel_first_pointer(again) == parts[0]
    again.close()
    want = []
    for layer in range(3):
        call(layer)
        att.sync()
        want.append(got[layer].clone())
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in range(2)]
    for rep in range(5):
        for t in got:
            t.zero_()
        torch.cuda.synchronize()
        for _ in range(10):
            for g, s in zip(graphs, streams):
                g.launch(s.cuda_stream)
            call(2)
        torch.cuda.synchronize()
        att.sync()
        for layer in range(3):
            assert torch.equal(got[layer].view(torch.int32), want[layer].view(torch.int32)), (rep, layer)
    for g in graphs:
        g.close()
    att.close()
