"""Attention over several 1024-key partitions: split across workgroups (few queries
over a long context) and merged inside one (many), the bits do not depend on which,
and both match the oracle."""
import numpy as np
import pytest

import jev
from helpers import worst_close
from oracle import oracle

pytestmark = pytest.mark.gpu

VOCAB = 2048
ROWS = [5, 77, 1999]


# 32 / 8 heads: tokens in all, of them new, workgroups that share a tile's output dims,
# partitions to a run
RUNS = [(2049, 200, 2, 1), (2700, 200, 1, 1), (4396, 30, 4, 1), (4396, 300, 1, 2), (12450, 250, 1, 4), (12200, 600, 1, 8)]


@pytest.mark.parametrize("total,new,ds,parts", RUNS)
def test_runs_of_several_partitions_give_the_whole_prompt_s_bits(gpu, total, new, ds, parts):
    # a workgroup whose run holds several partitions stores each one's partial as
    # it goes on to the next; the whole prompt merges them in its registers
    cfg = jev.ModelConfig(n_layers=1, hidden=256, n_heads=32, n_kv_heads=8, head_dim=128, ffn=512, vocab=VOCAB,
                          initial_kv_capacity=64)
    model = jev.SynthModel(cfg, jev.TYPE_Q8_0).open(0)
    tokens = jev.random_tokens(total, VOCAB, 22)
    outputs = [0, 1, new // 2, new - 2, new - 1]
    lay = jev.TokenLayout.tree(0, total, [], total).with_outputs([total - new + o for o in outputs])
    whole = model.forward_layout(tokens, lay, jev.OUT_FULL)
    model.kv_truncate(total - new)
    lay = jev.TokenLayout.tree(total - new, new, [], new).with_outputs(outputs)
    assert np.array_equal(whole, model.forward_layout(tokens[total - new:], lay, jev.OUT_FULL))
    model.close()


@pytest.mark.parametrize("heads,kv", [(4, 2), (6, 1), (32, 8)])
def test_suffix_bits_do_not_depend_on_the_split(gpu, heads, kv):
    # prompts whose last token sits around the partition edges: the same tokens as a
    # whole prompt (in-kernel merges or a split, by its size) and as suffixes of a
    # few tokens over the cached rest (split), with a token-level tail
    cfg = jev.ModelConfig(n_layers=1, hidden=256, n_heads=heads, n_kv_heads=kv, head_dim=128, ffn=512, vocab=VOCAB,
                          initial_kv_capacity=64)
    model = jev.SynthModel(cfg, jev.TYPE_Q8_0).open(0)
    tokens = jev.random_tokens(2700, VOCAB, 21)
    for n in (511, 512, 513, 514, 576, 577, 1023, 1024, 1025, 1088, 1089, 1600, 2049, 2700):
        model.reset_kv_cache()
        lay = jev.TokenLayout.tree(0, n, [], n).with_outputs([n - 40, n - 2, n - 1])
        whole = model.forward_layout(tokens[:n], lay, jev.OUT_FULL).reshape(3, VOCAB)
        for tail in (2, 33, 41, 200):
            model.kv_truncate(n - tail)
            lay = jev.TokenLayout.tree(n - tail, tail, [], tail).with_outputs([tail - 2, tail - 1])
            got = model.forward_layout(tokens[n - tail:n], lay, jev.OUT_FULL).reshape(2, VOCAB)
            assert np.array_equal(whole[1:], got), (n, tail)
    model.close()


def test_tree_over_a_long_cached_trunk_equals_the_whole_and_the_branches_alone(gpu):
    cfg = jev.ModelConfig(n_layers=2, hidden=256, n_heads=8, n_kv_heads=2, head_dim=128, ffn=512, vocab=VOCAB,
                          initial_kv_capacity=64)
    model = jev.SynthModel(cfg, jev.TYPE_Q5_1).open(0)
    trunk = jev.random_tokens(1530, VOCAB, 4)
    branches = [jev.random_tokens(n, VOCAB, 30 + n) for n in (3, 48, 70, 2)]
    whole = np.array(model.forward_tree(trunk, branches, ROWS))
    for cached in (500, 1024, 1529):
        model.kv_truncate(cached)
        assert np.array_equal(whole, np.array(model.forward_tree(trunk[cached:], branches, ROWS))), cached
    for i, b in enumerate(branches):
        model.kv_truncate(1530)
        assert np.array_equal(whole[i], np.array(model.forward_branches([b], ROWS))[0]), i
    model.close()


def test_partitioned_attention_matches_oracle(gpu):
    cfg = jev.ModelConfig(n_layers=2, hidden=256, n_heads=4, n_kv_heads=2, head_dim=128, ffn=512, vocab=VOCAB,
                          initial_kv_capacity=64)
    synth = jev.SynthModel(cfg, jev.TYPE_Q8_0)
    model, ref = synth.open(0), oracle.OracleModel(cfg).bind_synth(synth)
    tokens = jev.random_tokens(1400, VOCAB, 9)
    assert worst_close(ref.forward(tokens[:1100]), model.forward(tokens[:1100])) <= 1e-3
    assert worst_close(ref.forward(tokens[1100:1130]), model.forward(tokens[1100:1130])) <= 1e-3  # split
    assert worst_close(ref.forward(tokens[1130:]), model.forward(tokens[1130:])) <= 1e-3
    ref.close()
    model.close()
