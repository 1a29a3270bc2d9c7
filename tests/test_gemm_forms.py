"""Which tiles the GEMM takes above 512 rows at sizes that tests/test_gpu_tiles.py
compares, so that each height is known to be compared: without a device
(tests/fake_hip.py), from the launches."""
import fake_hip
import jev

FOUR, T64, T80, T96 = (4, 4, 4), (4, 2, 8), (5, 2, 8), (6, 2, 8)  # 16-row, 16-column tiles per wave, waves


def tiles(code):
    return [tuple(x) for x in fake_hip.run("""
import re
def tile(log, mode):
    for k, *_ in log:
        m = re.search(r"gemm_bd_kernelILi\\d+ELi%dELi(\\d)ELi(\\d)ELi1ELi\\dELb0ELi(\\d+)E" % mode, k)
        if m: return [int(v) for v in m.groups()]
result = []
""" + code)]


def test_every_height_of_a_store_is_compared():
    for t, block, want in [(jev.TYPE_Q4_0, 18, [T80, T96, FOUR, T96]), (jev.TYPE_Q8_0, 34, [T80, FOUR, FOUR, T96]),
                           (jev.TYPE_Q5_1, 24, [T80, T64, T64, T64])]:
        got = tiles(f"""
w = jev.QuantWeight({t}, 3060, 2112, np.zeros(3060 * 66 * {block}, np.uint8))
for n in (700, 900, 961, 1500):
    launches()
    w.matmul_device(4096, n, 8192)
    result.append(tile(launches(), 0))
""")
        assert got == want, t


def test_every_height_of_a_gated_projection_is_compared():
    for t, want in [(jev.TYPE_Q4_0, [T80, T96, T80, FOUR]), (jev.TYPE_Q8_0, [T80, T96, T80, FOUR]),
                    (jev.TYPE_Q5_1, [T80, T64, T80, T80])]:
        got = tiles(f"""
m = jev.SynthModel(jev.ModelConfig(n_layers=1, vocab=512, initial_kv_capacity=1100), {t}).open(0)
for n in (520, 576, 700, 1024):
    m.reset_kv_cache()
    launches()
    m.prefill(tokens(n))
    result.append(tile(launches(), 1))
""")
        assert got == want, t
