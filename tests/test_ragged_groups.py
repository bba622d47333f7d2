"""Element-wise maps and reductions over rows whose length or start is not a
multiple of four elements: groups of four read from any element address, the
last group of a row starting four before its end (it repeats elements the
group before has: a map stores the same bits twice, a sum skips them).

Maps of + - x are compared with the oracle bit for bit; sums within
n eps32 sum|x| (any order of fp32 additions); max and argmax exactly. The
C-ABI cases start at element offsets 1..3 of a buffer and check that nothing
outside the output is written."""
import ctypes

import numpy as np
import pytest
from conftest import fp32_sum_tolerance
from test_map_cabi import BF16, F32, Dev, make_desc, mapc  # noqa: F401

from ormi_amd import Tensor

# The smaller half stays below the size from which ragged rows take groups.
SHAPES = [(1, 5), (7, 7), (2, 1021), (129, 66), (2, 3, 5), (16384, 5), (9363, 7), (65, 1021), (1, 65537), (33, 2047), (32, 2049),
          (17, 4099), (1009, 66), (4099, 17), (4, 9, 2050), (16, 1025, 5)]


@pytest.mark.parametrize("shape", SHAPES + [(58543, 5), (5000, 301), (4000, 301), (5000, 401), (13948, 791), (4000, 791), (420, 163)])
def test_ragged_group_kernels_plan_vectors(ob, cpu, shape):
    """Ragged rows take groups of four from 256 x 4 x 64 elements up; a reduction's
    from 160 elements a row, and of many rows only those that keep its waves
    busy (no GPU)."""
    x, b = (Tensor(np.zeros(s, np.float32), "cpu") for s in (shape, shape[-1:]))
    rows, cols = int(np.prod(shape[:-1])), shape[-1]
    large = rows * cols >= 65536
    assert ("vec=4" if large else "vec=1") in ob._plan_kernel(((x + b) * 2.0)._node)["plan"]
    groups = large and cols >= 160 and (rows <= 4096 or not (256 < cols <= 384 or 768 < cols <= 1024))
    assert ("vec=4" if groups else "vec=1") in ob._plan_kernel(ob.sum(x._node, [len(shape) - 1], False))["plan"]


@pytest.mark.parametrize("shape,groups", [((16384, 129), True), ((33000, 65), True), ((33500, 63), False), ((16384, 127), False), ((47, 3251), False),
                                          ((1030, 2047), True), ((1100, 2049), False)])
def test_ragged_columns_plan_vectors(ob, cpu, shape, groups):
    """64 to 2048 ragged columns of 2^21 elements or more (no GPU)."""
    x = Tensor(np.zeros(shape, np.float32), "cpu")
    assert ("vec=4" if groups else "vec=1") in ob._plan_kernel(ob.sum(x._node, [0], False))["plan"]


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "bfloat16", "float16"])
@pytest.mark.parametrize("shape", SHAPES)
def test_ragged_maps_match_oracle(cpu, hip, shape, dtype):
    rng = np.random.default_rng(int(np.prod(shape)))
    x = rng.standard_normal(shape).astype(np.float32)
    bias = rng.standard_normal(shape[-1]).astype(np.float32)
    scale = rng.uniform(0.5, 1.5, shape[:-1] + (1,)).astype(np.float32)

    def graph(dev):
        X = Tensor(x, dev, dtype=dtype)
        z = (X + Tensor(bias, dev)) * Tensor(scale, dev) - X * 0.5
        return z, X * X - 1.0, z.astype(dtype)

    for got, want in zip(graph(hip), graph(cpu)):
        got, want = got.numpy(), want.numpy()
        assert got.dtype == want.dtype and np.array_equal(got, want)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("shape", SHAPES + [(5000, 5), (4099, 301), (70000, 17), (301, 4099), (66, 20001), (4200, 501), (2, 16384, 65)])
def test_ragged_reductions(hip, shape, dtype):
    rng = np.random.default_rng(int(np.prod(shape)) + 1)
    x = np.round(rng.standard_normal(shape) * 16).astype(np.float32) / 16  # exact in bfloat16, with ties
    X = Tensor(x, hip, dtype=dtype)
    for axis in range(len(shape)):
        got = X.sum(axis).numpy().astype(np.float64)
        assert np.all(np.abs(got - x.astype(np.float64).sum(axis)) <= fp32_sum_tolerance(x, axis))
        assert np.array_equal(X.max(axis).numpy(), x.max(axis))
        assert np.array_equal(X.argmax(axis).numpy(), x.argmax(axis))
        flat = Tensor(np.full(shape, -np.inf, np.float32), hip, dtype=dtype)
        assert np.array_equal(flat.argmax(axis).numpy(), np.zeros(x.max(axis).shape, np.int64))


@pytest.mark.gpu
@pytest.mark.parametrize("dtype,np_dtype", [(F32, np.uint32), (BF16, np.uint16)])
@pytest.mark.parametrize("shape", [(1, 9), (3, 64), (65, 1027), (32, 4096)])
@pytest.mark.parametrize("off_in,off_out", [(1, 0), (0, 1), (3, 2)])
def test_unaligned_buffers(mapc, hip, shape, dtype, np_dtype, off_in, off_out):  # noqa: F811
    """Negation (a sign-bit flip in any float type) between unaligned buffers."""
    n, es = int(np.prod(shape)), np.dtype(np_dtype).itemsize
    bits = np.random.default_rng(n).standard_normal(n).astype(np.float32).view(np.uint32)
    src = (bits if es == 4 else bits >> 16).astype(np_dtype)
    dev = Dev(mapc)
    try:
        pin, pout = dev.alloc((n + 8) * es), dev.alloc((n + 8) * es)
        assert mapc.ormi_hip_memcpy_h2d(ctypes.c_void_p(pin + off_in * es), src.ctypes.data, n * es) == 0
        guard = np.full(n + 8, 0xA5A5 if es == 2 else 0xA5A5A5A5, np_dtype)
        assert mapc.ormi_hip_memcpy_h2d(ctypes.c_void_p(pout), guard.ctypes.data, (n + 8) * es) == 0
        d, keep = make_desc(shape, [(pin + off_in * es, dtype, False, (shape[1], 1))], [("NEG", 0, 0, F32)],
                            [(1, pout + off_out * es, dtype)])
        assert mapc.ormi_hip_map(ctypes.byref(d)) == 0
        got = dev.get(pout, (n + 8) * es).view(np_dtype)
    finally:
        dev.free()
    want = guard.copy()
    want[off_out:off_out + n] = src ^ np_dtype(1 << (8 * es - 1))
    assert np.array_equal(got, want)
