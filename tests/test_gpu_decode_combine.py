"""One token over a long context has its attention chunks combined ahead of the O
projection, over a short one inside it: the same bits on both sides of the change,
which goes by the longest context a decode may reach."""
import numpy as np
import pytest

import jev
from helpers import tiny_config

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
