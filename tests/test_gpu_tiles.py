"""Every tile shape the GEMM dispatch picks from (by rows and by the width of the
weight) gives a row the same bits: windows of rows at the sizes where the choice
changes, against the same rows of one large call, over a weight that ends inside
a 16-row group and K splits of unequal length; and, through a one-layer model at
the 3B widths, the fused QKV and SwiGLU projections, whose tiles a matmul call
does not reach, by a causal prompt's early tokens at growing prompt lengths."""
import numpy as np
import pytest

import jev
from test_gpu_kernels import matmul_gpu

pytestmark = pytest.mark.gpu

TYPES = [jev.TYPE_Q4_0, jev.TYPE_Q5_1, jev.TYPE_Q8_0]


@pytest.mark.parametrize("t", TYPES)
@pytest.mark.parametrize("rows", [3060, 1000])
def test_matmul_rows_do_not_depend_on_the_tile_shape(gpu, t, rows):
    cols = 2112  # 66 quant blocks: splits of 18, 18, 18 and 12
    raw = jev.synth_tensor("tiles", t, rows, cols)
    x = np.random.default_rng(2).standard_normal((800, cols)).astype(np.float32)
    full = matmul_gpu(t, raw, rows, cols, x, 800)
    for n in (16, 17, 32, 33, 48, 49, 64, 65, 96, 97, 128, 129, 160, 161, 192, 193, 256, 257, 320, 512, 513, 640, 641):
        lo = (n * 7) % (800 - n)
        assert np.array_equal(full[lo:lo + n], matmul_gpu(t, raw, rows, cols, x[lo:lo + n], n)), n


@pytest.mark.parametrize("t", TYPES)
def test_prompt_rows_do_not_depend_on_the_prompt_length(gpu, t):
    cfg = jev.ModelConfig(n_layers=1, vocab=2048, initial_kv_capacity=1024)
    model = jev.SynthModel(cfg, t).open(0)
    tokens = jev.random_tokens(700, cfg.vocab, 3)
    seen = None
    for n in (700, 17, 32, 48, 49, 64, 96, 97, 128, 129, 160, 161, 192, 193, 224, 225, 256, 257, 288, 320, 321, 384, 448,
              449, 512, 513, 640):
        model.reset_kv_cache()
        lay = jev.TokenLayout.tree(0, n, [], n).with_outputs([2, 9, 16])
        got = model.forward_layout(tokens[:n], lay, jev.OUT_FULL)
        if seen is None:
            seen = got
        assert np.array_equal(seen, got), n
    model.close()


@pytest.mark.parametrize("t", TYPES)
def test_matmul_rows_do_not_depend_on_the_height_of_a_large_batch_tile(gpu, t):
    rows, cols = 3060, 2112
    raw = jev.synth_tensor("tall", t, rows, cols)
    x = np.random.default_rng(6).standard_normal((1700, cols)).astype(np.float32)
    full = matmul_gpu(t, raw, rows, cols, x, 1700)
    # 80-row tiles at 700, 96-row ones at 1500 (Q5_1: 64-row), 64-row or four-wave ones between
    for n in (641, 700, 720, 721, 768, 900, 960, 961, 1100, 1500, 1536, 1537):
        lo = (n * 7) % (1700 - n)
        assert np.array_equal(full[lo:lo + n], matmul_gpu(t, raw, rows, cols, x[lo:lo + n], n)), n


@pytest.mark.parametrize("t", TYPES)
def test_prompt_rows_do_not_depend_on_a_longer_prompt_s_tiles(gpu, t):
    cfg = jev.ModelConfig(n_layers=1, vocab=512, initial_kv_capacity=1100)
    model = jev.SynthModel(cfg, t).open(0)
    tokens = jev.random_tokens(1024, cfg.vocab, 8)
    seen = None
    for n in (17, 520, 560, 561, 576, 700, 720, 900, 960, 961, 1024):
        model.reset_kv_cache()
        got = model.forward_layout(tokens[:n], jev.TokenLayout.tree(0, n, [], n).with_outputs([2, 9, 16]), jev.OUT_FULL)
        seen = got if seen is None else seen
        assert np.array_equal(seen, got), n
    model.close()
