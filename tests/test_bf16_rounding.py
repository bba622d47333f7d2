"""float32 to bfloat16 (ormi_f32_to_bf16, one gfx950 instruction): nearest even,
NaN a quiet NaN with its upper payload, subnormals kept. Every one of the 2^32
inputs through the conversion entry; the generated kernels' cast over every
upper half with the lower halves around each rounding boundary."""
import ctypes

import numpy as np
import pytest
from test_map_cabi import BF16, F32, Dev

from ormi_amd import Tensor

LOWS = np.array([0, 1, 2, 0x3FFF, 0x4000, 0x7FFE, 0x7FFF, 0x8000, 0x8001, 0x8002, 0xC000, 0xFFFE, 0xFFFF], np.uint32)


def rounded(high, low):
    """The 16 bits for each upper half (rows) and lower half (columns)."""
    high, low = high.astype(np.uint16)[:, None], low[None, :]
    up = [low > 0x8000, low >= 0x8000]  # even, odd upper half
    out = high + np.where(high & 1, up[1], up[0]).astype(np.uint16)
    nan = (high[:, 0] & 0x7F80) == 0x7F80
    out[nan] = np.where((high[nan] & 0x7F != 0) | (low != 0), high[nan] | 0x40, high[nan])
    return out


def test_rounded_against_known_values():
    """The reference of these tests on values anyone can check (no GPU)."""
    high = np.array([0x3F80, 0x3F81, 0x7F7F, 0x7F80, 0xFF80, 0x7F81, 0x0000], np.uint32)
    got = rounded(high, np.array([0, 1, 0x8000, 0x8001], np.uint32))
    want = [[0x3F80, 0x3F80, 0x3F80, 0x3F81], [0x3F81, 0x3F81, 0x3F82, 0x3F82], [0x7F7F, 0x7F7F, 0x7F80, 0x7F80],
            [0x7F80, 0x7FC0, 0x7FC0, 0x7FC0], [0xFF80, 0xFFC0, 0xFFC0, 0xFFC0], [0x7FC1, 0x7FC1, 0x7FC1, 0x7FC1], [0, 0, 0, 1]]
    assert got.tolist() == want


@pytest.mark.gpu
def test_every_float32(hip, cabi):
    step, low = 2048, np.arange(1 << 16, dtype=np.uint32)
    dev = Dev(cabi)
    src, dst = dev.alloc(step << 18), dev.alloc(step << 17)
    bits = np.empty((step, 1 << 16), np.uint32)
    got = np.empty((step, 1 << 16), np.uint16)
    try:
        for first in range(0, 1 << 16, step):
            high = np.arange(first, first + step, dtype=np.uint32)
            np.bitwise_or(high[:, None] << 16, low, out=bits)
            assert cabi.ormi_hip_memcpy_h2d(ctypes.c_void_p(src), bits.ctypes.data, bits.nbytes) == 0
            assert cabi.ormi_hip_convert(ctypes.c_void_p(dst), BF16, ctypes.c_void_p(src), F32, bits.size) == 0
            assert cabi.ormi_hip_memcpy_d2h(got.ctypes.data, ctypes.c_void_p(dst), got.nbytes) == 0
            assert np.array_equal(got, rounded(high, low)), hex(first)
    finally:
        dev.free()


@pytest.mark.gpu
def test_generated_cast(hip, cabi):
    high = np.arange(1 << 16, dtype=np.uint32)
    x = ((high[:, None] << 16) | LOWS).view(np.float32)
    t = Tensor(x, hip).astype("bfloat16").realize()
    got = np.empty(x.shape, np.uint16)
    assert cabi.ormi_hip_memcpy_d2h(got.ctypes.data, ctypes.c_void_p(t._node.data.ptr), got.nbytes) == 0
    assert np.array_equal(got, rounded(high, LOWS))
