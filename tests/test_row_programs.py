"""Row programs: several reductions over the rows of one shape, the
element-wise values around them and column sums, as one kernel that reads each
operand once (backend/hip/rows.cpp, plan_rows in codegen.cpp).

Row layouts covered: fewer lanes than a wave per row, one wave, several waves
sharing a row through LDS, rows that are not a multiple of four elements, rows
shorter than four, a last partial set of rows, more rows than work-groups, and
rows too long for the registers (realized one by one as before).

Sums are checked against float64 within n eps32 sum|v| (any order of fp32
additions), maxima and argmax exactly (ties, NaN and -inf among the values)."""
import ctypes
import threading

import numpy as np
import pytest
from conftest import fp32_sum_tolerance
from test_cabi_codegen import _compile_only

from ormi_amd import Tensor, realize_all

EPS32 = float(np.finfo(np.float32).eps)
SHAPES = [(2, 2), (5, 3), (40, 72), (70, 301), (300, 17), (4099, 16), (50000, 7), (33, 1024), (129, 1028), (700, 2049), (64, 2500),
          (1000, 1536), (301, 8192), (3, 30000), (20, 16383), (5, 7, 130), (6, 3, 5)]


def values(shape, seed=0):
    """Sixteenths, so that ties are common and sums of a few hundred are exact."""
    rng = np.random.default_rng(int(np.prod(shape)) + seed)
    return np.round(rng.standard_normal(shape) * 32).astype(np.float32) / 16


def stats(x):
    last, lead = len(x.shape) - 1, list(range(len(x.shape) - 1))
    top = x.max(last, keepdims=True)
    return top, (x - top).exp().sum(last), x.mean(last), x.argmax(last), x.sum(lead)


def softmax(x):
    last = len(x.shape) - 1
    e = (x - x.max(last, keepdims=True)).exp()
    return e / e.sum(last, keepdims=True)


@pytest.mark.parametrize("shape", [(40, 72), (70, 301), (129, 1028), (300, 8192), (20, 16383), (5, 7, 130), (5, 3)])
def test_programs_compile(ob, cpu, cabi, shape):
    """One kernel for the row statistics (two with the column sums' finish) and
    one for a softmax, for every row layout (no GPU)."""
    x = Tensor(np.zeros(shape, np.float32), "cpu")
    for nodes, two in ((stats(x), True), (stats(x)[:4], False), ([softmax(x)], False)):
        d = ob._plan_rows([t._node for t in nodes])
        assert d is not None and d["two_pass"] == two and d["plan"].startswith("rows"), d
        for src in [d["source"]] + ([d["second_source"]] if two else []):
            rc, _ = _compile_only(cabi, src, ob._rtc_options())
            assert rc == 0, (d["plan"], cabi.ormi_hip_last_error())


def test_what_is_no_program(ob, cpu):
    """One reduction (with its prologue or scale), unrelated operands, another
    axis, a single row, and rows too long for the registers."""
    x, y = (Tensor(np.ones((8, 64), np.float32), "cpu") for _ in range(2))

    def plan(*t):
        return ob._plan_rows([u._node for u in t])

    assert plan((x * 2.0).sum(1)) is None and plan(x.mean(1)) is None
    assert plan(x.sum(1), y.max(1)) is None
    assert plan(x.sum(1), x.sum(1)) is not None
    assert plan(x.max(1), x.sum([0, 1])) is None
    one = Tensor(np.ones((1, 64), np.float32), "cpu")
    assert plan(one.sum(1), one.max(1)) is None
    wide = Tensor(np.ones((2, 40000), np.float32), "cpu")
    assert plan(wide.sum(1), wide.max(1)) is None


DEEP = 60000


def deep(kind, x):
    """Roots over a chain of DEEP nodes."""
    h = x.max(1, keepdims=True) if kind == "views" else x
    for i in range(DEEP):
        if kind == "reductions":
            if i % 4 == 0:  # four nodes a level
                h = h - h.max(1, keepdims=True) * 0.5
        elif kind == "views":
            h = h.reshape(h.shape[:1] if i % 2 == 0 else (h.shape[0], 1))
        else:
            h = h + 1.0
    return {"maps": lambda: [h.sum(1), h.max(1)], "beside": lambda: [x.sum(1), h], "softmax": lambda: [softmax(h)],
            "reductions": lambda: [h], "views": lambda: [x - h]}[kind]()


@pytest.mark.parametrize("kind", ["maps", "beside", "softmax", "reductions", "views"])
def test_deep_chains_are_declined_on_a_small_stack(ob, cpu, kind):
    """A chain of any length is looked at as far as a program could reach, not
    to its end: a thread of 256 KB has the stack for it."""
    roots = [t._node for t in deep(kind, Tensor(np.ones((8, 64), np.float32), "cpu"))]
    found = []
    old = threading.stack_size(256 << 10)
    try:
        t = threading.Thread(target=lambda: found.append(ob._plan_rows(roots)))
        t.start()
    finally:
        threading.stack_size(old)
    t.join()
    assert found == [None]


def of_indices(i, j, x):
    """Values computed from the indices i and j of rows of x."""
    return [i / j, i * 0.5, i.astype("float32") + x.max(1), x - i.reshape((x.shape[0], 1)).astype("float32")]


def test_an_argmax_is_no_operand(ob, cpu):
    """What reads an ARGMAX of the program is not part of it: the kernel holds
    the index as an integer."""
    x = Tensor(values((40, 72)), "cpu")
    i, j = x.argmax(1), (-x).argmax(1)
    assert ob._plan_rows([i._node, j._node]) is not None
    for q in of_indices(i, j, x):
        assert ob._plan_rows([i._node, j._node, q._node]) is None


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(40, 72), (70, 301), (3, 2049)])
def test_values_of_an_argmax_beside_it(hip, shape):
    """The same results realized with the indices as without: a quotient is not
    truncated, and one by index 0 is inf or NaN."""
    x = values(shape, 4)
    x[0, 0], x[1, 0], x[2, 1] = 9.0, -9.0, 9.0
    X = Tensor(x, hip)
    i, j = X.argmax(1), (-X).argmax(1)
    got = of_indices(i, j, X)
    realize_all(i, j, *got)
    a, b = x.argmax(1), (-x).argmax(1)
    assert np.array_equal(i.numpy(), a) and np.array_equal(j.numpy(), b) and a[0] == 0 and b[1] == 0
    a32, b32 = a.astype(np.float32), b.astype(np.float32)
    with np.errstate(divide="ignore", invalid="ignore"):
        np.testing.assert_allclose(got[0].numpy(), a32 / b32, rtol=4 * EPS32)
    for t, want in zip(got[1:], (a32 * np.float32(0.5), a32 + x.max(1), x - a32[:, None])):
        assert np.array_equal(t.numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", ["float32", "bfloat16"])
@pytest.mark.parametrize("shape", SHAPES)
def test_stats(ob, hip, shape, dtype):
    x = values(shape)  # exact in bfloat16 below 8
    x = np.clip(x, -7.5, 7.5)
    got = stats(Tensor(x, hip, dtype=dtype))
    before = ob._kernel_launches()
    realize_all(*got)
    assert ob._kernel_launches() - before == 2
    top, denom, mean, arg, cols = (t.numpy() for t in got)
    last, lead = len(shape) - 1, tuple(range(len(shape) - 1))
    x6 = x.astype(np.float64)
    assert np.array_equal(top, x.max(last, keepdims=True)) and np.array_equal(arg, x.argmax(last))
    e = np.exp(x6 - x6.max(last, keepdims=True))
    assert np.all(np.abs(denom - e.sum(last)) <= (shape[-1] + 4) * EPS32 * e.sum(last))
    assert np.all(np.abs(mean - x6.mean(last)) <= fp32_sum_tolerance(x, last) / shape[-1] + EPS32 * np.abs(x6.mean(last)))
    assert cols.shape == x.sum(lead).shape and np.all(np.abs(cols - x6.sum(lead)) <= fp32_sum_tolerance(x, lead))


@pytest.mark.gpu
def test_waves_of_a_row_add_pairwise(ob, hip):
    """Sixteen waves share a row, one group of four per lane: 2 + 6 + 4 levels of
    additions, each off by at most half an ulp of the row's sum. One wave's sum
    after the other would lose all fifteen ones against 2^24."""
    x = np.zeros((8, 4096), np.float32)
    x[:, 256::256] = 1.0
    x[:, 0] = 2.0 ** 24
    X = Tensor(x, hip)
    s, top = X.sum(1), X.max(1)
    assert "lanes=1024 groups=1" in ob._plan_rows([s._node, top._node])["plan"]
    realize_all(s, top)
    exact = x.astype(np.float64).sum(1)
    assert np.all(np.abs(s.numpy() - exact) <= 12 * EPS32 / 2 * exact) and np.all(top.numpy() == 2.0 ** 24)


@pytest.mark.gpu
def test_column_sums_of_work_groups_add_pairwise(ob, hip):
    """One row per work-group, so 256 parts per column: 4 + 4 levels of additions,
    each off by at most half an ulp of the column's sum. One part after the other
    would lose the fifteen ones of the first wave's parts against 2^24, one wave
    after the other the fifteen of the other waves."""
    x = np.zeros((256, 4096), np.float32)
    x[1:16], x[16::16] = 1.0, 1.0
    x[0] = 2.0 ** 24
    X = Tensor(x, hip)
    s, top = X.sum(0), X.max(1)
    assert "O=256 R=4096 vec=4 lanes=256" in ob._plan_rows([s._node, top._node])["plan"]
    realize_all(s, top)
    exact = x.astype(np.float64).sum(0)
    assert np.all(np.abs(s.numpy() - exact) <= 8 * EPS32 / 2 * exact) and np.all(top.numpy() == x.max(1))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_special_values(hip, shape):
    """Rows of -inf only, with inf, and with NaN: the first NaN is the maximum."""
    x = values(shape, 1)
    flat = x.reshape(-1, shape[-1])
    flat[0] = -np.inf
    flat[1, shape[-1] // 2] = np.nan
    flat[1, -1] = np.nan
    flat[-1, 0] = np.inf if len(flat) > 2 else flat[-1, 0]
    X, last = Tensor(x, hip), len(shape) - 1
    top, arg, both = X.max(last), X.argmax(last), (X * X).max(last)
    realize_all(top, arg, both)
    with np.errstate(invalid="ignore"):
        assert np.array_equal(top.numpy(), x.max(last), equal_nan=True)
        assert np.array_equal(arg.numpy(), x.argmax(last))
        assert np.array_equal(both.numpy(), (x * x).max(last), equal_nan=True)


@pytest.mark.gpu
@pytest.mark.parametrize("shape", SHAPES)
def test_softmax(ob, hip, shape):
    x = values(shape, 2)
    y = softmax(Tensor(x, hip))
    before = ob._kernel_launches()
    y.realize()
    assert ob._kernel_launches() - before == 1
    x6 = x.astype(np.float64)
    e = np.exp(x6 - x6.max(-1, keepdims=True))
    want = e / e.sum(-1, keepdims=True)
    assert np.all(np.abs(y.numpy() - want) <= (shape[-1] + 8) * EPS32 * want + 1e-44)


@pytest.mark.gpu
@pytest.mark.parametrize("cast", [None, "bfloat16"])
@pytest.mark.parametrize("shape", [s for s in SHAPES if s[-1] >= 16])
def test_normalization_forward_and_backward(ob, hip, shape, cast):
    """Full outputs, column sums and per-row values in one program. Absolute
    bounds in units of what is summed: c eps32 times the row length's sqrt
    amplifies nothing here (unit-variance rows), so a few hundred eps32."""
    rng = np.random.default_rng(shape[-1])
    x, dy = (rng.standard_normal(shape).astype(np.float32) for _ in range(2))
    gamma, beta = rng.uniform(0.5, 1.5, shape[-1:]).astype(np.float32), rng.standard_normal(shape[-1:]).astype(np.float32)
    X, G, B = (Tensor(a, hip, requires_grad=True) for a in (x, gamma, beta))
    last, lead = len(shape) - 1, tuple(range(len(shape) - 1))
    c = X - X.mean(last, keepdims=True)
    inv = ((c * c).mean(last, keepdims=True) + 1e-5) ** -0.5
    y = c * inv * G + B
    total = (y * Tensor(dy, hip)).sum()
    total.backward()
    out = [y if cast is None else y.astype(cast), X.grad, G.grad, B.grad]
    realize_all(*out)
    y, gx, gg, gb = (t.numpy() for t in out)
    total.zero_grad_graph()
    x6, dy6 = x.astype(np.float64), dy.astype(np.float64)
    c6 = x6 - x6.mean(-1, keepdims=True)
    i6 = 1 / np.sqrt((c6 * c6).mean(-1, keepdims=True) + 1e-5)
    u, g6 = c6 * i6, dy6 * gamma
    rows = np.prod(shape[:-1])
    tol = 64 * EPS32 * (1 + i6)  # small rows can have a small spread
    assert np.all(np.abs(y - (u * gamma + beta)) <= (tol if cast is None else tol + 2.0 ** -8 * np.abs(u * gamma + beta)) * (1 + np.abs(u)))
    assert np.all(np.abs(gx - i6 * (g6 - g6.mean(-1, keepdims=True) - u * (g6 * u).mean(-1, keepdims=True)))
                  <= tol * (1 + i6) * (1 + np.abs(u)) * (4 + np.abs(g6)))
    assert np.all(np.abs(gg - (dy6 * u).sum(lead)) <= (rows + 64) * EPS32 * (np.abs(dy6) * (1 + np.abs(u)) * (1 + i6)).sum(lead))
    assert np.all(np.abs(gb - dy6.sum(lead)) <= fp32_sum_tolerance(dy, lead))


@pytest.mark.gpu
def test_operands_of_every_kind(hip):
    """Broadcast rows and columns, a transposed operand (one-element groups), a
    scalar, a partial broadcast over the leading dims, and a reduction's result
    used by a later program."""
    rng = np.random.default_rng(7)
    a = rng.standard_normal((6, 50, 33)).astype(np.float32)
    t = rng.standard_normal((33, 50, 6)).astype(np.float32)
    row, col, part = (rng.standard_normal(s).astype(np.float32) for s in ((33,), (6, 50, 1), (6, 1, 33)))
    A, Tt, Rw, Cl, Pt = (Tensor(v, hip) for v in (a, t, row, col, part))
    z = A * Cl + Rw - Tt.transpose() * Pt
    z = z - z.mean(2, keepdims=True)
    scale = (z * z).sum(2, keepdims=True)
    w = z / (scale + 1.0)
    realize_all(w, scale)
    again = (z * scale).sum(2)  # scale holds a buffer now
    z6 = a.astype(np.float64) * col + row - t.T.astype(np.float64) * part
    z6 = z6 - z6.mean(2, keepdims=True)
    s6 = (z6 * z6).sum(2, keepdims=True)
    np.testing.assert_allclose(w.numpy(), z6 / (s6 + 1), rtol=0, atol=64 * EPS32 * np.abs(z6).max())
    np.testing.assert_allclose(scale.numpy(), s6, rtol=64 * EPS32)
    assert np.all(np.abs(again.numpy() - (z6 * s6).sum(2)) <= 64 * EPS32 * (np.abs(z6) * s6 + s6).sum(2))


@pytest.mark.gpu
def test_deep_chain_of_rows(hip):
    """Longer than one program holds: cut, without recursion per level."""
    x = values((16, 64), 3)
    X, want = Tensor(x, hip), x.copy()
    for _ in range(200):
        X = X - X.max(1, keepdims=True) * 0.5
        want = want - want.max(1, keepdims=True) * np.float32(0.5)
    assert np.array_equal(X.numpy(), want)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["maps", "beside", "reductions"])
def test_deep_chains_realize(hip, kind):
    """DEEP nodes, one root or two: cut into programs and kernels without
    recursion per level."""
    x = values((8, 64), 6)
    roots = deep(kind, Tensor(x, hip))
    realize_all(*roots)
    # 1.0 added DEEP times to sixteenths of magnitude below 8 is exact.
    if kind == "reductions":
        want = x.copy()
        for _ in range(0, DEEP, 4):
            want = want - want.max(1, keepdims=True) * np.float32(0.5)
        assert np.array_equal(roots[0].numpy(), want)
    elif kind == "maps":
        h = x + np.float32(DEEP)
        assert np.array_equal(roots[1].numpy(), h.max(1))
        assert np.all(np.abs(roots[0].numpy() - h.astype(np.float64).sum(1)) <= 64 * EPS32 * h.sum(1))
    else:
        assert np.array_equal(roots[1].numpy(), x + np.float32(DEEP))
        assert np.all(np.abs(roots[0].numpy() - x.astype(np.float64).sum(1)) <= fp32_sum_tolerance(x, 1))


@pytest.mark.gpu
def test_a_gradient_owns_its_buffer(hip, cabi):
    """1 * w as a gradient is a copy of w, asked for first, last or after the
    products that read w in its place: filling it leaves w as it was."""
    rng = np.random.default_rng(8)
    a, b, w = (rng.standard_normal(s).astype(np.float32) for s in ((40, 24), (24, 56), (40, 56)))
    W, nine = Tensor(w, hip), np.array([9], np.float32)

    def fill(t):
        assert np.array_equal(t.numpy(), w) and t._node.data.ptr != W._node.data.ptr
        assert cabi.ormi_hip_fill(ctypes.c_void_p(t._node.data.ptr), nine.ctypes.data, 4, w.size) == 0
        assert np.array_equal(t.numpy(), np.full_like(w, 9)) and np.array_equal(W.numpy(), w)

    X = Tensor(w * 2, hip, requires_grad=True)
    (X * W).sum().backward()
    fill(X.grad)
    for first in (True, False):
        A, B = Tensor(a, hip, requires_grad=True), Tensor(b, hip, requires_grad=True)
        C = A @ B
        total = (C * W).sum()
        total.backward()
        if first:
            realize_all(C.grad, A.grad, B.grad)
        else:
            realize_all(A.grad, B.grad)
        assert np.all(np.abs(A.grad.numpy() - w.astype(np.float64) @ b.T) <= 60 * EPS32 * (np.abs(w) @ np.abs(b).T))
        assert np.all(np.abs(B.grad.numpy() - a.T.astype(np.float64) @ w) <= 60 * EPS32 * (np.abs(a).T @ np.abs(w)))
        fill(C.grad)
        total.zero_grad_graph()


@pytest.mark.gpu
def test_a_seed_times_a_buffer_is_the_buffer(ob, hip):
    """The gradient of sum(c * w) with respect to c is w: no kernel copies it, and
    the two backward products read it as it is; a transposed or broadcast w is
    still multiplied out."""
    rng = np.random.default_rng(5)
    a, b, w = (rng.standard_normal(s).astype(np.float32) for s in ((40, 24), (24, 56), (40, 56)))
    for wt in (Tensor(w, hip), Tensor(np.ascontiguousarray(w.T), hip).transpose(), Tensor(w[:1], hip)):
        A, B = Tensor(a, hip, requires_grad=True), Tensor(b, hip, requires_grad=True)
        total = ((A @ B) * wt).sum()
        total.backward()
        before = ob._kernel_launches()
        realize_all(A.grad, B.grad)
        if wt.op == ob.OpEnum.LEAF and wt.shape == (40, 56):
            assert ob._kernel_launches() == before
        full = np.broadcast_to(w[:1], w.shape) if wt.shape == (1, 56) else w
        for got, want, scale in ((A.grad, full.astype(np.float64) @ b.T, np.abs(full) @ np.abs(b).T),
                                 (B.grad, a.T.astype(np.float64) @ full, np.abs(a).T @ np.abs(full))):
            assert np.all(np.abs(got.numpy() - want) <= 60 * EPS32 * scale)
        total.zero_grad_graph()
