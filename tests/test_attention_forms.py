"""Which form of the attention kernels the GPU tests' shapes take, so that each form is
known to be compared: without a device (tests/fake_hip.py), from the launches."""
import fake_hip
from test_gpu_attn_partitions import RUNS
from test_gpu_decode_shared_lds import FEW, SHAPES
from test_gpu_model import TREE_FORMS


def test_tree_passes_and_their_branches():
    got = fake_hip.run(f"""
m = model(4, 2, cap=16384)
result = []
for trunk in {list(TREE_FORMS)}:
    m.reset_kv_cache()
    launches()
    m.forward_tree(tokens(trunk), [tokens(40), tokens(3)], [1])
    result.append(attention(launches())[:3])
    for n in (40, 3):
        m.kv_truncate(trunk)
        launches()
        m.forward(tokens(n))
        result.append(attention(launches())[1])
""")
    assert [tuple(g) for g in got[::3]] == list(TREE_FORMS.values())
    forms = {f[:2] for f in TREE_FORMS.values()}
    assert forms >= {(4, "one"), (2, "merged"), (1, "merged"), (2, "split"), (1, "split")}
    # at 6000 and 12000 split branches meet a merged tree and runs of two partitions
    assert got[1::3] == got[2::3] == ["one", "merged"] + ["split"] * 5


def test_runs_of_one_and_several_partitions():
    got = fake_hip.run(f"""
m = model(cap=16384)
result = []
for total, new, ds, parts in {RUNS}:
    m.reset_kv_cache()
    m.prefill(tokens(total))
    whole = attention(launches())
    m.kv_truncate(total - new)
    launches()
    m.prefill(tokens(new))
    result.append([whole, attention(launches())])
    launches()
""")
    for (total, new, ds, parts), (whole, split) in zip(RUNS, got):
        assert whole == [1, "merged", 1, False]
        partitions = -(-total // 1024)
        assert split == [ds, "split", ds * -(-partitions // parts), True], (total, new)
    assert {r[3] for r in RUNS} >= {1, 2, 4, 8} and {r[2] for r in RUNS} == {1, 2, 4}


def test_decode_attention_with_v_behind_k():
    got = fake_hip.run(f"""
result = []
for heads, kv, rows, keys in {SHAPES}:
    length = [keys - 37 * r for r in range(rows)]
    base = jev.row_bases(length, 8)
    m = model(heads, kv, cap=32768)
    for n in (rows, {FEW}):
        launches()
        m.forward_rows(0, base[:n], length[:n], [[1]] * n, [1])
        result.append(["attn_decode_kernelILb1E" in k for k, g, a, b in launches() if "attn_decode_kernel" in k])
""")
    assert got == [[True], [False]] * len(SHAPES)
