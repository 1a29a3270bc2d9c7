"""The split attention's partials are scratch that only makes a pass faster: where
the device has no room for them the pass runs whole, and where another allocation
has no room beside them they are given back.  Without a device (tests/fake_hip.py):
which allocations and launches the calls make."""
import pytest

import fake_hip


def test_a_pass_without_room_for_its_partials_runs_whole():
    # 450 tokens over 12000 cached take 99 MiB of partials
    got = fake_hip.run("""
m = model()
m.prefill(tokens(12000))
launches()
result = []
for left in (40 * MIB, 0, None):
    room(left)
    m.kv_truncate(12000)
    logits = m.forward(tokens(450))
    result.append([attention(launches())[1:], m.cached_token_count, logits.size])
""")
    whole, split = ["merged", 2, False], ["split", 13, True]
    assert got == [[whole, 12450, 512], [whole, 12450, 512], [split, 12450, 512]]


@pytest.mark.parametrize("what,need", [
    ("m.prefill(tokens(5000))", "4 * 8 * 32768 * 512"),            # the KV cache doubled
    ("snap = m.kv_snapshot_device(12000)", "2 * 8 * 12000 * 512"),  # a snapshot
    ("m.kv_truncate(0); m.forward_layout(tokens(12100), jev.TokenLayout.tree(0, 12100, [], 12100)"
     ".with_outputs(list(range(12100))), jev.OUT_FULL)", "12100 * 512 * 4"),  # logits
    ("m.kv_truncate(0); m.forward_rows(0, [0, 6100], [0, 0], [tokens(6100), tokens(6100)])", "1 << 16"),  # activations
    ("m.decode_greedy(1, 3)", "1"),
    ("m.decode_rows_greedy(0, [13000, 14000], [0, 0], [1, 2], 20)", "1"),
])
def test_an_allocation_without_room_takes_the_partials_back(what, need):
    # after a split pass (99 MiB of partials), with a byte less than the call allocates
    got = fake_hip.run(f"""
m = model()
m.prefill(tokens(12000))
m.prefill(tokens(450))
m.kv_truncate(12000)
launches()
room({need} - 1)
{what}
result = [F.fake_refused(), len(launches())]
""")
    assert got[0] == 1, got  # one refusal, and the call went on


def test_a_call_that_fits_keeps_the_partials():
    got = fake_hip.run("""
m = model()
m.prefill(tokens(12000))
live = []
for n in (450, 450, 300):
    m.kv_truncate(12000)
    m.forward(tokens(n))
    live.append(F.fake_live())
result = [live, F.fake_refused()]
""")
    assert got[0][0] == got[0][1] == got[0][2] and got[1] == 0
