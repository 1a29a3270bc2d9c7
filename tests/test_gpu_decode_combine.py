"""One token over a long context has its attention chunks combined ahead of the O
projection, over a short one inside it: the same bits on both sides of the change,
which goes by the longest context a decode may reach; and contexts of more chunks
than the combining kernel takes at a time, against the chunks merged on the host."""
import numpy as np
import pytest

import jev
import npref
from helpers import tiny_config, worst_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("t", [jev.TYPE_Q4_0, jev.TYPE_Q5_1, jev.TYPE_Q8_0])
@pytest.mark.parametrize("cached", [200, 1022, 1023, 1024, 2100])
def test_decode_tokens_do_not_depend_on_where_the_chunks_are_combined(gpu, t, cached):
    # 16 chunks of 64 keys are the last combined inside; steps of one token choose by
    # their own length, a longer run by its end
    synth = jev.SynthModel(tiny_config(initial_kv_capacity=64), t)
    tokens = jev.random_tokens(cached, synth.config.vocab, 5)
    with synth.open(0) as m:
        m.prefill(tokens)
        want, tok = [], 7
        for _ in range(4):
            tok = int(m.decode_greedy(tok, 1)[0])
            want.append(tok)
        last = m.forward([tok])
        m.kv_truncate(cached)
        got = m.decode_greedy(7, 4)
        assert np.array_equal(got, want)
        assert np.array_equal(last, m.forward([tok]))
        m.kv_truncate(cached)
        assert np.array_equal(m.decode_greedy(7, 2200)[:4], want)  # combined from the first step
        m.kv_truncate(cached + 4)  # whose cache rows give the step behind them the same bits
        assert np.array_equal(last, m.forward([tok]))


@pytest.mark.parametrize("t", [jev.TYPE_Q4_0, jev.TYPE_Q5_1, jev.TYPE_Q8_0])
@pytest.mark.parametrize("cached", [1100, 4094, 4096, 4160, 8300])
def test_combined_chunks_over_long_contexts(gpu, t, cached):
    # The combining kernel takes 64 chunks (4096 keys) at a time: contexts on both sides
    # of the second round, and a third one.  attn_weighted is the chunks merged on the
    # host, attn_out the O projection of what the kernel made of them.  Of the n chunks'
    # terms each is off by its exponential (a few ulp) and its turn in the chain, in all
    # (n + 8) 2^-23 of their size, at most max |v|; the projection's fp16 pairs, 32-term
    # products and up to 16 block sums are off by 2^-18 of its terms.
    synth = jev.SynthModel(tiny_config(initial_kv_capacity=64), t)
    c = synth.config
    tokens = jev.random_tokens(cached + 1, c.vocab, 6)
    with synth.open(0) as m:
        m.prefill(tokens[:cached])
        taps = dict(m.forward_capture(tokens[cached:])[1])
        vmax = float(np.abs(m.kv_snapshot(cached + 1)).max())
        m.kv_truncate(cached)
        one = m.forward(tokens[cached:])
        m.kv_truncate(cached - 1)
        two = m.forward(tokens[cached - 1:])  # tree attention, GEMMs
    weights, n = npref.dequantized(synth), (cached + 64) // 64
    for layer in range(c.n_layers):
        w = weights["blk.%d.attn_output.weight" % layer]
        x = taps["blk.%d.attn_weighted" % layer].reshape(-1).astype(np.float64)
        off = np.abs(taps["blk.%d.attn_out" % layer].reshape(-1) - w @ x)
        assert np.all(off <= np.abs(w) @ (2.0 ** -18 * np.abs(x) + (n + 8) * 2.0 ** -23 * vmax)), layer
    assert worst_close(two, one) <= 1e-3
