"""The tiles a Q5_1 weight is repacked into on the host, field by field, against the
GGUF blocks' own quants: 16 rows x two blocks per tile, whole and ragged."""
import ctypes

import numpy as np
import pytest

import jev

ROWS, COLS, THREADS = [1, 16, 33, 70], [32, 64, 160], 3


@pytest.mark.parametrize("rows", ROWS)
@pytest.mark.parametrize("cols", COLS)
def test_every_field_holds_the_blocks_quants(rows, cols):
    raw = np.random.default_rng(rows * cols).integers(0, 256, (rows, cols // 32, 24), dtype=np.uint8)
    groups, pairs = -(-rows // 16), -(-(cols // 32) // 2)
    n = groups * pairs
    at, sizes = [0], [512 * n, 128 * n, 128 * n, 1024 * n]  # words, scales and mins, low bits, bytes
    for s in sizes:
        at.append(-(-(at[-1] + s) // 256) * 256)
    out = np.full(at[4], 0xA5, np.uint8)
    repack = jev.lib()._ZN3jev11repack_hostEillPKvPvi
    repack.restype = ctypes.c_bool
    repack.argtypes = [ctypes.c_int, ctypes.c_int64, ctypes.c_int64, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int]
    assert repack(jev.TYPE_Q5_1, rows, cols, raw.ctypes.data, out.ctypes.data, THREADS)

    # the quants of the blocks [row][block][32], zero past the weight
    nib = np.concatenate([raw[:, :, 8:] & 15, raw[:, :, 8:] >> 4], 2)
    fifth = np.unpackbits(raw[:, :, 4:8], axis=2, bitorder="little")
    q = np.zeros((groups * 16, pairs * 2, 32), np.uint32)
    q[:rows, :cols // 32] = nib | fifth << 4
    dm = np.zeros((groups * 16, pairs * 2, 2), np.uint16)
    dm[:rows, :cols // 32] = np.ascontiguousarray(raw[:, :, :4]).view(np.uint16)
    # [group][pair][g][row][block][8]: lane 16 g + row, its block bb, k = 8 g .. 8 g + 7
    q = q.reshape(groups, 16, pairs, 2, 4, 8).transpose(0, 2, 4, 1, 3, 5)
    dm = dm.reshape(groups, 16, pairs, 2, 2).transpose(0, 2, 1, 4, 3)  # row's two scales, then its two mins

    def field(i):
        return out[at[i]:at[i] + sizes[i]]

    word = sum(q[..., i] << (5 * (i // 2) + 16 * (i % 2)) for i in range(6)) | (q[..., 6] >> 4) << 15 | (q[..., 7] >> 4) << 31
    assert np.array_equal(field(0).view(np.uint32), word.ravel().astype(np.uint32))
    assert np.array_equal(field(1).view(np.uint16), dm.ravel())
    low = (q[..., 6:] & 15).astype(np.uint8)  # [..., block, element 6 | 7]
    assert np.array_equal(field(2), (low[..., 0, :] | low[..., 1, :] << 4).ravel())
    assert np.array_equal(field(3), q.astype(np.uint8).ravel())
