"""Kernels at the edges of their tiles and dispatch ranges, each against the CPU
oracle: partial tiles and stages, the smallest and odd sizes, both sides of each
rule that picks a kernel."""
import numpy as np
import pytest

import oracle as O
from gpu_util import assert_bits_equal
from proj_cases import make_bias, make_rows

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
