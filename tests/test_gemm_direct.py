"""Products by register fragments loaded straight from memory
(gemm_direct.hip): the sizes where tiles, fragments and k-steps end (1, 15..17,
31..33, 63..65 and the like), every pair of layouts and types, unaligned bases
and row strides, K shares that leave waves without a step, splits across
work-groups, batches with a broadcast operand, and every epilogue, in place too.

Bound: the componentwise error of a length-K fp32 accumulation in any order, of
products that are exact in fp32 for 16-bit operands and rounded once for fp32:
(K + 2) eps32 (|A| |B|); an epilogue adds its own few roundings."""
import ctypes

import numpy as np
import pytest
from test_gemm_epilogue import Epi
from test_map_cabi import Dev

EPS32 = float(np.finfo(np.float32).eps)
F32, BF16, F16 = 0, 3, 4


class Desc(ctypes.Structure):
    _fields_ = [("dtype", ctypes.c_int), ("M", ctypes.c_int), ("N", ctypes.c_int), ("K", ctypes.c_int),
                ("a", ctypes.c_void_p), ("a_stride_m", ctypes.c_int64), ("a_stride_k", ctypes.c_int64),
                ("b", ctypes.c_void_p), ("b_stride_k", ctypes.c_int64), ("b_stride_n", ctypes.c_int64),
                ("c", ctypes.c_void_p), ("batch_ndim", ctypes.c_int), ("batch_shape", ctypes.c_int * 4),
                ("a_batch_stride", ctypes.c_int64 * 4), ("b_batch_stride", ctypes.c_int64 * 4)]


def storage(x, dtype):
    """x's bits in dtype and the float64 values they hold."""
    if dtype == F32:
        return x, x.astype(np.float64)
    if dtype == F16:
        h = x.astype(np.float16)
        return h, h.astype(np.float64)
    u = x.view(np.uint32)
    h = ((u + 0x7FFF + ((u >> 16) & 1)) >> 16).astype(np.uint16)
    return h, (h.astype(np.uint32) << 16).view(np.float32).astype(np.float64)


class Product:
    """Operands in padded buffers (row pitch = extent + pad, base shifted by
    `shift` elements) so that nothing but the element size is aligned."""

    def __init__(self, lib, dtype, layout, M, N, K, batch=1, share_b=False, pad=0, shift=0, seed=0):
        self.lib, self.dev, self.M, self.N, self.K, self.batch = lib, Dev(lib), M, N, K, batch
        rng = np.random.default_rng(seed + M * 7 + N * 3 + K)
        es = 4 if dtype == F32 else 2

        def operand(rows, cols, count):
            x = rng.standard_normal((count, rows, cols)).astype(np.float32)
            bits, val = storage(x, dtype)
            buf = np.zeros((count, rows, cols + pad), bits.dtype)
            buf[:, :, :cols] = bits
            raw = np.concatenate([np.zeros(shift, bits.dtype), buf.reshape(-1)])
            p = self.dev.alloc(raw.nbytes)
            assert lib.ormi_hip_memcpy_h2d(ctypes.c_void_p(p), raw.ctypes.data, raw.nbytes) == 0
            return p + shift * es, val, cols + pad, rows * (cols + pad)

        ta, tb = layout[0] == "t", layout[1] == "t"
        pa, va, lda, sa = operand(*((K, M) if ta else (M, K)), batch)
        pb, vb, ldb, sb = operand(*((N, K) if tb else (K, N)), 1 if share_b else batch)
        self.A = va.transpose(0, 2, 1) if ta else va
        self.B = vb.transpose(0, 2, 1) if tb else vb
        d = self.d = Desc(dtype=dtype, M=M, N=N, K=K, a=pa, b=pb)
        d.a_stride_m, d.a_stride_k = (1, lda) if ta else (lda, 1)
        d.b_stride_k, d.b_stride_n = (1, ldb) if tb else (ldb, 1)
        if batch > 1:
            d.batch_ndim, d.batch_shape[0], d.a_batch_stride[0], d.b_batch_stride[0] = 1, batch, sa, 0 if share_b else sb
        self.exact = self.A @ self.B
        self.bound = (K + 2) * EPS32 * (np.abs(self.A) @ np.abs(self.B)) + 1e-30
        self.n = batch * M * N
        d.c = self.c = self.put(np.full(self.n + 4, 7.0, np.float32))

    def put(self, x):
        p = self.dev.alloc(x.nbytes)
        assert self.lib.ormi_hip_memcpy_h2d(ctypes.c_void_p(p), x.ctypes.data, x.nbytes) == 0
        return p

    def get(self, p=None):
        raw = self.dev.get(p or self.c, (self.n + 4) * 4).view(np.float32)
        if p is None:
            assert np.all(raw[self.n:] == 7.0)  # nothing past the output
        return raw[:self.n].reshape(self.batch, self.M, self.N)

    def run(self, epi=None):
        rc = self.lib.ormi_hip_gemm_ex(ctypes.byref(self.d), ctypes.byref(epi) if epi else None)
        assert rc == 0, self.lib.ormi_hip_last_error()

    def check(self, got, want=None, extra=0.0):
        want = self.exact if want is None else want
        assert np.all(np.abs(got - want) <= self.bound * (1 + extra) + extra * EPS32 * (1 + np.abs(want)))


@pytest.fixture(params=["by size", "always"])
def product(cabi, request, monkeypatch):
    """By size: the kernels that the dispatch takes. Always: those of
    gemm_direct.hip wherever they can run (ORMI_GEMM_DIRECT, read per call)."""
    monkeypatch.setenv("ORMI_GEMM_DIRECT", "1" if request.param == "by size" else "2")
    made = []

    def make(*a, **k):
        made.append(Product(cabi, *a, **k))
        return made[-1]

    yield make
    for p in made:
        p.dev.free()


SIZES = [(1, 4, 1), (1, 1, 5), (3, 3, 40), (1, 5, 31), (4, 1, 33), (15, 64, 32), (16, 65, 33), (17, 63, 95), (16, 4097, 160), (12, 1000, 2049),
         (33, 31, 127), (65, 17, 300), (61, 1690, 49), (64, 64, 4096), (100, 130, 70), (200, 1003, 205), (500, 16, 513), (1001, 1003, 45)]


@pytest.mark.gpu
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("dtype", [F32, BF16, F16])
def test_sizes(hip, product, dtype, layout):
    for M, N, K in SIZES:
        p = product(dtype, layout, M, N, K)
        p.run()
        p.check(p.get())


@pytest.mark.gpu
@pytest.mark.parametrize("pad,shift", [(0, 1), (1, 0), (3, 3)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("dtype", [F32, BF16, F16])
def test_unaligned_operands(hip, product, dtype, layout, pad, shift):
    for M, N, K in [(16, 64, 64), (40, 96, 128), (256, 128, 96), (2, 4, 65)]:
        p = product(dtype, layout, M, N, K, pad=pad, shift=shift)
        p.run()
        p.check(p.get())


@pytest.mark.gpu
@pytest.mark.parametrize("share_b", [False, True])
@pytest.mark.parametrize("dtype,layout", [(F16, "nt"), (F32, "nn"), (BF16, "tn")])
def test_batches(hip, product, dtype, layout, share_b):
    for b, M, N, K in [(3, 50, 33, 65), (48, 19, 70, 30), (2, 16, 700, 1000)]:
        p = product(dtype, layout, M, N, K, batch=b, share_b=share_b)
        p.run()
        p.check(p.get())


@pytest.mark.gpu
def test_non_finite_values_stay_in_their_rows(hip, product, cabi):
    """inf and NaN past a row's or the k-range's end reach no other element: the
    last partial k-step and the clamped rows must not multiply them in."""
    for dtype, layout in [(F32, "nn"), (BF16, "nn"), (F16, "tn"), (F32, "nt")]:
        M, N, K = 18, 70, 37
        p = product(dtype, layout, M, N, K, pad=5)
        ta, tb = layout[0] == "t", layout[1] == "t"
        es = 4 if dtype == F32 else 2
        nan = {F32: np.uint32(0x7FC00000), BF16: np.uint16(0x7FC0), F16: np.uint16(0x7E00)}[dtype]
        pads = np.full(5, nan)
        for base, rows, ld, cols in ((p.d.a, K if ta else M, (M if ta else K) + 5, M if ta else K),
                                     (p.d.b, N if tb else K, (K if tb else N) + 5, K if tb else N)):
            for r in range(rows):
                assert cabi.ormi_hip_memcpy_h2d(ctypes.c_void_p(base + (r * ld + cols) * es), pads.ctypes.data, pads.nbytes) == 0
        p.run()
        p.check(p.get())


@pytest.mark.gpu
@pytest.mark.parametrize("M,N,K", [(12, 1000, 2049), (33, 31, 127), (61, 1690, 49), (300, 70, 500)])
@pytest.mark.parametrize("dtype", [F32, BF16])
def test_epilogues(hip, product, dtype, M, N, K):
    rng = np.random.default_rng(3)
    D = rng.standard_normal((M, N)).astype(np.float32)
    s = np.float32(-0.37)
    p = product(dtype, "nn", M, N, K)
    d, ps = p.put(np.concatenate([D.reshape(-1), np.zeros(4, np.float32)])), p.put(np.array([s], np.float32))
    v = p.exact[0]
    for form, want in ((0, D + v * s), (1, D - v * s), (2, v * s - D)):
        p.run(Epi(kind=1, form=form, s=ps, d=d, d_stride_m=N, d_stride_n=1))
        p.check(p.get()[0], want, 4.0)
    aux = p.put(np.full(p.n + 4, 7.0, np.float32))
    p.run(Epi(kind=2, fn=1, aux=aux))
    p.check(p.get()[0], np.maximum(v, 0))
    p.check(p.get(aux)[0], v)
    p.run(Epi(kind=3, fn=0, d=d, d_stride_m=N, d_stride_n=1))
    assert np.all(np.abs(p.get()[0] - v * D) <= (p.bound[0] + EPS32 * np.abs(v)) * np.abs(D) * 1.01 + 1e-30)
    # In place: each element's D is read before its product is stored there.
    p2 = product(dtype, "nn", M, N, K)
    start = np.concatenate([D.reshape(-1), np.full(4, 7.0, np.float32)])
    assert p2.lib.ormi_hip_memcpy_h2d(ctypes.c_void_p(p2.c), start.ctypes.data, start.nbytes) == 0
    p2.run(Epi(kind=1, form=1, s=ps, d=p2.c, d_stride_m=N, d_stride_n=1))
    p2.check(p2.get()[0], D - p2.exact[0] * s, 4.0)


# ------------------------------------------------- activation and its cast --
def test_cast_entry_checks_its_arguments(cabi):
    d, e = Desc(dtype=BF16, M=4, N=4, K=4, a=256, a_stride_m=4, a_stride_k=1, b=512, b_stride_k=4, b_stride_n=1, c=1024), Epi(kind=2, fn=7)

    def call(desc=d, epi=e, cast=2048, dtype=BF16):
        return cabi.ormi_hip_gemm_ex_cast(ctypes.byref(desc), ctypes.byref(epi) if epi else None, ctypes.c_void_p(cast), dtype)

    f32 = Desc.from_buffer_copy(d)
    f32.dtype = F32
    assert call(desc=f32) == 3 and call(epi=None) == 3 and call(epi=Epi(kind=1, d=256)) == 3
    assert call(cast=None) == 3 and call(cast=2049) == 3 and call(dtype=F32) == 3


@pytest.mark.gpu
@pytest.mark.parametrize("fn", ["gelu", "relu", "tanh", "sigmoid"])
@pytest.mark.parametrize("dtype", ["bfloat16", "float16"])
@pytest.mark.parametrize("M,K,N", [(12, 512, 1000), (5, 333, 77), (256, 1024, 512), (300, 2048, 2048), (3, 40, 7)])
def test_activation_and_its_cast_from_one_product(ob, hip, M, K, N, dtype, fn):
    """The rounded activation comes from the GEMM, with the bits of the separate
    cast, and the product and the activation hold their buffers as well."""
    from ormi_amd import Tensor

    rng = np.random.default_rng(M + N)
    x = Tensor(rng.standard_normal((M, K)).astype(np.float32), hip, dtype=dtype)
    w = Tensor((rng.standard_normal((K, N)) / 16).astype(np.float32), hip, dtype=dtype)
    p = x @ w
    act = getattr(p, fn)()
    h = act.astype(dtype)
    before = ob._kernel_launches()
    h.realize()
    assert ob._kernel_launches() == before and p._node.is_realized and act._node.is_realized
    q = (x @ w).realize()
    act2 = getattr(q, fn)().realize()
    assert np.array_equal(p.numpy(), q.numpy()) and np.array_equal(act.numpy(), act2.numpy())
    assert np.array_equal(h.numpy(), act2.astype(dtype).numpy())


@pytest.mark.gpu
@pytest.mark.parametrize("cast_dtype", [BF16, F16])
@pytest.mark.parametrize("dtype", [BF16, F16])
@pytest.mark.parametrize("batch,M,N,K,layout,step", [
    (3, 50, 33, 65, "nt", 1),      # direct, one pass
    (2, 16, 700, 4096, "nn", 1),   # direct, split over K: the finish pass
    (3, 17, 40, 31, "nn", 2),      # no unit stride, small: the generic kernel
    (2, 200, 320, 300, "nn", 2),   # no unit stride, packed: the tiles and the finish pass
    (2, 64, 256, 4096, "nt", 1),   # the tiles and the finish pass
])
def test_cast_of_a_batch_is_laid_out_like_c(hip, product, cabi, dtype, cast_dtype, batch, M, N, K, layout, step):
    """Every matrix of the batch has its own rounded values, bit for bit those
    of C, and nothing is written past the last."""
    p = product(dtype, layout, M, N, K * step, batch=batch)
    if step > 1:  # every step-th k of A
        p.d.K, p.d.a_stride_k = K, step
        a, b = p.A[:, :, ::step], p.B[:, :K]
        p.exact, p.bound = a @ b, (K + 2) * EPS32 * (np.abs(a) @ np.abs(b)) + 1e-30
    aux, out = p.put(np.full(p.n + 4, 7.0, np.float32)), p.put(np.full(p.n + 8, 0x1234, np.uint16))
    e = Epi(kind=2, fn=1, aux=aux)
    rc = cabi.ormi_hip_gemm_ex_cast(ctypes.byref(p.d), ctypes.byref(e), ctypes.c_void_p(out), cast_dtype)
    assert rc == 0, cabi.ormi_hip_last_error()
    c = p.get()
    p.check(p.get(aux))
    p.check(c, np.maximum(p.exact, 0))
    got = p.dev.get(out, (p.n + 8) * 2).view(np.uint16)
    assert np.array_equal(got[:p.n], storage(c.reshape(-1), cast_dtype)[0].view(np.uint16)) and np.all(got[p.n:] == 0x1234)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [F32, BF16, F16])
def test_generic_kernel_adds_in_short_chains(hip, cabi, monkeypatch, dtype):
    """K = 96 in six steps of four chains of four: 3 + 2 + 6 additions after the
    largest term, 2^24, each off by at most half an ulp, 1. One chain through K
    would lose all 95 ones."""
    monkeypatch.setenv("ORMI_GEMM_DIRECT", "0")
    M, N, K = 3, 5, 96
    p = Product(cabi, dtype, "nn", M, N, K)
    try:
        a, b = np.ones((M, K), np.float32), np.ones((K, N), np.float32)
        a[:, 0], b[0] = 2.0 ** 12, 2.0 ** 12
        for dst, x in ((p.d.a, a), (p.d.b, b)):
            bits = np.ascontiguousarray(storage(x, dtype)[0])
            assert cabi.ormi_hip_memcpy_h2d(ctypes.c_void_p(dst), bits.ctypes.data, bits.nbytes) == 0
        p.run()
        assert np.all(np.abs(p.get().astype(np.float64) - (2.0 ** 24 + K - 1)) <= 11)
    finally:
        p.dev.free()
