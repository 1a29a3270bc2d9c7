"""Calls of 2 to 16 rows take their own GEMM, whose workgroups' width and weight
reading go by the number of columns: every form of it gives a row the bits that a
larger call gives it, at column counts on both sides of each change, with odd and
unfilled K stages; and through a one-layer model for the SwiGLU forms (with the
Q5_1 block sums and without)."""
import numpy as np
import pytest

import jev
from test_gpu_kernels import matmul_gpu

pytestmark = pytest.mark.gpu

TYPES = [jev.TYPE_Q4_0, jev.TYPE_Q5_1, jev.TYPE_Q8_0]


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("rows,cols", [(200, 96), (1000, 2112), (4112, 800), (16384, 224), (16400, 352), (24592, 224),
                                       (32784, 352), (65536, 96), (65537, 416)])
def test_few_rows_match_a_larger_call(gpu, t, rows, cols):
    raw = jev.synth_tensor("few", t, rows, cols)
    x = np.random.default_rng(5).standard_normal((33, cols)).astype(np.float32)
    full = matmul_gpu(t, raw, rows, cols, x, 33)
    for lo, n in ((0, 2), (7, 5), (20, 12), (17, 16)):
        assert np.array_equal(full[lo:lo + n], matmul_gpu(t, raw, rows, cols, x[lo:lo + n], n)), n


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("ffn", [448, 8192, 8256, 12352])
def test_few_tokens_match_a_longer_prompt(gpu, t, ffn):
    cfg = jev.ModelConfig(n_layers=1, vocab=512, ffn=ffn, initial_kv_capacity=64)
    model = jev.SynthModel(cfg, t).open(0)
    tokens = jev.random_tokens(40, cfg.vocab, 4)
    seen = None
    for n in (40, 3, 8, 16):
        model.reset_kv_cache()
        got = model.forward_layout(tokens[:n], jev.TokenLayout.tree(0, n, [], n).with_outputs([0, 1, 2]), jev.OUT_FULL)
        seen = got if seen is None else seen
        assert np.array_equal(seen, got), n
    model.close()
