"""The per-kernel profiler times every attention launch: the tree attention with a
split pass's merge, the decode attention with the combination of its chunks.  Without
a device (tests/fake_hip.py), from the events the launches carry; every launch there
takes 1 ms."""
import pytest

import fake_hip


@pytest.mark.parametrize("call,kernels,cls", [
    ("m.prefill(tokens(450))", ["attn_tree_kernel", "attn_merge_kernel"], "PROF_ATTN"),
    ("m.kv_truncate(0); m.prefill(tokens(2000))", ["attn_tree_kernel"], "PROF_ATTN"),  # whole tiles
    ("m.forward([1])", ["attn_decode_kernel", "attn_combine_one_kernel"], "PROF_DECODE_ATTN"),
    ("m.kv_truncate(300); m.forward([1])", ["attn_decode_kernel"], "PROF_DECODE_ATTN"),  # combined in the O projection
    ("m.decode_greedy(1, 1)", ["attn_decode_kernel", "attn_combine_one_kernel"], "PROF_DECODE_ATTN"),
    ("m.decode_rows_greedy(0, [13000, 14000], [0, 0], [1, 2], 1)", ["attn_decode_kernel", "attn_combine_kernel"],
     "PROF_DECODE_ATTN"),
])
def test_attention_launches_are_stamped(call, kernels, cls):
    log, read = fake_hip.run(f"""
m = model()
m.prefill(tokens(12000))
L = jev.lib()
jev._lib.check(L.jev_profile_enable(m._h, 1))
launches()
{call}
n, ms = ctypes.c_int64(), ctypes.c_double()
jev._lib.check(L.jev_profile_read(m._h, jev._lib.{cls}, ctypes.byref(n), ctypes.byref(ms), None, None))
result = [[(k, a, b) for k, g, a, b in launches() if "attn_" in k], [n.value, ms.value]]
""")
    assert len(log) == len(kernels) and all(k in name for k, (name, _, _) in zip(kernels, log)), log
    assert all(a and b and a != b for _, a, b in log), log
    assert read == [len(kernels), float(len(kernels))]
