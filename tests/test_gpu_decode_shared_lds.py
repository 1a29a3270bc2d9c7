"""The decode attention of more than 512 workgroups lets V follow K into the same LDS:
a row among many gives the bits that it gives among few, for groups of two, three and
four query heads, with chunks that are full and not."""
import numpy as np
import pytest

import jev

pytestmark = pytest.mark.gpu

# heads, KV heads, rows of the large pass (KV heads x chunks x rows workgroups), keys of the longest
SHAPES = [(32, 8, 12, 660), (32, 8, 7, 640), (24, 8, 12, 650), (16, 8, 12, 1100), (4, 2, 16, 1090)]
FEW = 3


@pytest.mark.parametrize("heads,kv,rows,keys", SHAPES)
def test_a_row_among_many_equals_the_row_among_few(gpu, heads, kv, rows, keys):
    cfg = jev.ModelConfig(n_layers=2, hidden=256, n_heads=heads, n_kv_heads=kv, head_dim=128, ffn=512, vocab=2048,
                          initial_kv_capacity=64)
    length = [keys - 37 * r for r in range(rows)]
    base = jev.row_bases(length, 8)
    last = [int(t) for t in jev.random_tokens(rows, 2048, 3)]
    with jev.SynthModel(cfg, jev.TYPE_Q5_1).open(0) as m:
        for r in range(rows):
            m.forward_rows(0, [base[r]], [0], [jev.random_tokens(length[r], 2048, 40 + r)], [1])
        many = m.forward_rows(0, base, length, [[t] for t in last])
        for r in range(0, rows - FEW + 1, 2):
            few = m.forward_rows(0, base[r:r + FEW], length[r:r + FEW], [[t] for t in last[r:r + FEW]])
            assert np.array_equal(many[r:r + FEW], few), r
        # as a graph over several steps
        tokens = m.decode_rows_greedy(0, base, length, last, 5)
        few = m.decode_rows_greedy(0, base[:FEW], length[:FEW], last[:FEW], 5)
        assert np.array_equal(tokens[:, :FEW], few)
