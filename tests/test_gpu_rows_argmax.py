"""The rows step's argmax takes its row in slices by the number of rows (32 for few,
one from 512): the graph's tokens are the step loop's first largest logits, at
vocabularies that are and are not whole 16-byte loads, in slices and per row."""
import numpy as np
import pytest

import jev
from helpers import tiny_config
from test_gpu_reasoning import _rows_stepwise

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [64, 2048, 2053])
@pytest.mark.parametrize("n_rows", [2, 16, 17, 40, 512, 513])
def test_rows_argmax_is_the_step_loop(gpu, vocab, n_rows):
    steps = 3
    synth = jev.SynthModel(tiny_config(vocab=vocab, initial_kv_capacity=64), jev.TYPE_Q8_0)
    first = [int(t) for t in jev.random_tokens(n_rows, vocab, 7)]
    bases = [8 * r for r in range(n_rows)]
    with synth.open(0) as m:
        got = m.decode_rows_greedy(0, bases, [0] * n_rows, first, steps)
        m.reset_kv_cache()
        want = _rows_stepwise(m, 0, bases, [0] * n_rows, first, steps)
    assert np.array_equal(got, want)
