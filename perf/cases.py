"""The work a program has this library do, as cases that can be timed and checked.

A case is a dict of plain values; prepare() builds what a program holds before
the call (tensors on the "hip" device), run() is one pass through the public
Tensor API, exact() the same outputs in 64 bits by plain torch. Eight kinds:

  rows_train  y = sum(relu(a*b + c) * 0.5, axis=1) and the gradients of sum(y)
              with respect to a, b, c: a fused element-wise and reduction step,
              forward and backward
  chain       tanh((x + bias) * scale) * sigmoid(x) - 0.1 x^2 with a bias row
              and a scale column: a broadcast element-wise chain, with x and
              the result in float32 or bfloat16
  stats       per row the maximum, the softmax denominator sum(exp(x - max)),
              the mean and the argmax, and the column sums of one tensor
  norm        layer normalization, forward and backward: y and the gradients
              of x, gamma and beta
  gemm        one product in bfloat16, float16 or float32, plain, with a
              transposed operand, or over a batch of matrices
  gemm_grad   a float32 product, forward and both backward products
  mlp_train   a training step of a three-layer GELU network: mean squared
              error, backward and the SGD update of every weight, float32
  mlp_infer   the forward pass of a three-layer GELU network with bfloat16
              weights at a small batch: the logits

The sizes of the listed cases are the benchmark's configurations (1024 x 1024
rows_train, 8192 x 4096 chain, 16384 x 8192 stats, 4096^3 bfloat16 product,
2048 x 1024 x 4096 float32 product with its backward, 1024-4096-4096-1024
network) and generic small, ragged and narrow ones.
"""
from __future__ import annotations

import ctypes
import math
from pathlib import Path

import numpy as np
import torch

import ormi_amd
from ormi_amd import Tensor, realize_all

_LIB = ctypes.CDLL(str(Path(ormi_amd.__file__).resolve().parent / "lib" / "libormi_hip.so"))
_LIB.ormi_hip_event_record.argtypes = [ctypes.c_void_p]
_LIB.ormi_hip_event_create.argtypes = [ctypes.POINTER(ctypes.c_void_p)]

LR = 1e-3  # SGD step of mlp_train
EPS = 1e-5  # layer normalization


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # The smallest call: host work and launches are all of it.
        {"name": "rows_train_small", "kind": "rows_train", "rows": 40, "cols": 72},
        # The benchmark's fused row reduction with its gradients.
        {"name": "rows_train", "kind": "rows_train", "rows": 1024, "cols": 1024},
        # The benchmark's broadcast chain.
        {"name": "chain", "kind": "chain", "rows": 8192, "cols": 4096, "dtype": "float32"},
        # An odd shape in the 16-bit type: no row starts on a vector boundary.
        {"name": "chain_ragged_bf16", "kind": "chain", "rows": 6001, "cols": 2047, "dtype": "bfloat16"},
        # The benchmark's row statistics of a large tensor.
        {"name": "stats", "kind": "stats", "rows": 16384, "cols": 8192},
        # Many short rows of an odd length (class scores, features of samples).
        {"name": "stats_narrow", "kind": "stats", "rows": 50021, "cols": 301},
        # A normalization layer's forward and backward at a model's width.
        {"name": "norm", "kind": "norm", "rows": 4095, "cols": 1536},
        # The benchmark's bfloat16 product.
        {"name": "gemm_bf16", "kind": "gemm", "dtype": "bfloat16", "layout": "nn", "batch": 1, "m": 4096, "n": 4096, "k": 4096},
        # A batch of small ragged products with a transposed operand: pairwise
        # scores of 197 vectors of 64 features in each of 48 groups.
        {"name": "gemm_batched_f16", "kind": "gemm", "dtype": "float16", "layout": "nt", "batch": 48, "m": 197, "n": 197, "k": 64},
        # The benchmark's float32 product and its two backward products.
        {"name": "gemm_grad", "kind": "gemm_grad", "m": 2048, "n": 4096, "k": 1024},
        # The benchmark's training step.
        {"name": "mlp_train", "kind": "mlp_train", "rows": 1024, "d0": 1024, "d1": 4096, "d2": 4096, "d3": 1024},
        # Serving a handful of requests: each weight is read once for 12 rows.
        {"name": "mlp_infer", "kind": "mlp_infer", "rows": 12, "d0": 2048, "d1": 8192, "d2": 4096, "d3": 1000},
    ]


def _log(rng, lo, hi, step=1):
    """A whole number of [lo, hi], spread over its logarithm."""
    return min(hi, max(lo, step * round(math.exp(rng.uniform(math.log(lo), math.log(hi))) / step)))


def draw(rng):
    kind = rng.choice(["rows_train", "chain", "stats", "norm", "gemm", "gemm_grad", "mlp_train", "mlp_infer"])
    step = rng.choice([1, 1, 8, 64])  # half of the sizes are odd or arbitrary, the others multiples
    if kind == "rows_train":
        return {"kind": kind, "rows": _log(rng, 16, 4096), "cols": _log(rng, 16, 4096, step)}
    if kind == "chain":
        return {"kind": kind, "rows": _log(rng, 64, 8192), "cols": _log(rng, 64, 4096, step),
                "dtype": rng.choice(["float32", "bfloat16"])}
    if kind == "stats":
        cols = _log(rng, 16, 16384, step)
        return {"kind": kind, "rows": _log(rng, 64, min(262144, (1 << 27) // cols)), "cols": cols}
    if kind == "norm":
        return {"kind": kind, "rows": _log(rng, 64, 16384), "cols": _log(rng, 64, 4096, step)}
    if kind == "gemm":
        dtype = rng.choice(["bfloat16", "float16", "float32"])
        case = {"kind": kind, "dtype": dtype, "layout": rng.choice(["nn", "nt", "tn"])}
        if rng.random() < 0.4:
            return {**case, "batch": _log(rng, 4, 96), "m": _log(rng, 16, 512, step), "n": _log(rng, 16, 512, step),
                    "k": _log(rng, 32, 512, step)}
        top = 2048 if dtype == "float32" else 4096
        return {**case, "batch": 1, "m": _log(rng, 32, top, step), "n": _log(rng, 32, top, step), "k": _log(rng, 32, top, step)}
    if kind == "gemm_grad":
        return {"kind": kind, "m": _log(rng, 32, 2048, step), "n": _log(rng, 32, 4096, step), "k": _log(rng, 32, 1024, step)}
    if kind == "mlp_train":
        return {"kind": kind, "rows": _log(rng, 16, 1024), "d0": _log(rng, 32, 1024, step), "d1": _log(rng, 64, 4096, step),
                "d2": _log(rng, 64, 4096, step), "d3": _log(rng, 10, 1024)}
    return {"kind": kind, "rows": _log(rng, 1, 64), "d0": _log(rng, 256, 4096, step), "d1": _log(rng, 256, 8192, step),
            "d2": _log(rng, 256, 8192, step), "d3": _log(rng, 10, 4096)}


# ------------------------------------------------------------------ inputs --
def _inputs(case, seed):
    """The case's inputs as host float32 arrays, in the order its pass reads them."""
    rng = np.random.default_rng(seed)
    kind = case["kind"]

    def normal(shape, scale=1.0):
        a = rng.standard_normal(shape, dtype=np.float32)
        a *= np.float32(scale)
        return a

    def uniform(shape, lo, hi):
        a = rng.random(shape, dtype=np.float32)
        a *= np.float32(hi - lo)
        a += np.float32(lo)
        return a

    if kind in ("rows_train", "chain", "stats", "norm"):
        r, c = case["rows"], case["cols"]
        if kind == "rows_train":
            return [uniform((r, c), -1, 1) for _ in range(3)]
        if kind == "chain":
            return [normal((r, c)), normal((c,), 0.1), uniform((r, 1), 0.5, 1.5)]
        if kind == "stats":
            return [normal((r, c), 2.0)]
        return [normal((r, c)), uniform((c,), 0.5, 1.5), normal((c,), 0.1), normal((r, c))]  # x, gamma, beta, dy
    if kind in ("gemm", "gemm_grad"):
        m, n, k = case["m"], case["n"], case["k"]
        lead = (case["batch"],) if case.get("batch", 1) > 1 else ()
        layout = case.get("layout", "nn")
        a = normal(lead + ((k, m) if layout == "tn" else (m, k)), 1 / 64)
        b = normal(lead + ((n, k) if layout == "nt" else (k, n)), 1 / 64)
        return [a, b] + ([normal((m, n))] if kind == "gemm_grad" else [])
    d = [case["d0"], case["d1"], case["d2"], case["d3"]]
    ws = [uniform((i, o), -math.sqrt(6 / i), math.sqrt(6 / i)) for i, o in zip(d, d[1:])]
    x = normal((case["rows"], d[0]))
    return [x] + ws + ([normal((case["rows"], d[3]))] if kind == "mlp_train" else [])


def _dtype(case, i):
    """Element type of input i on the device."""
    if case["kind"] == "chain":
        return case["dtype"] if i == 0 else "float32"
    return "bfloat16" if case["kind"] == "mlp_infer" else case.get("dtype", "float32")


def _trained(case, i):
    """Whether input i takes a gradient."""
    return {"rows_train": i < 3, "norm": i < 3, "gemm_grad": i < 2, "mlp_train": 1 <= i <= 3}.get(case["kind"], False)


def prepare(case, seed):
    event = ctypes.c_void_p()
    if _LIB.ormi_hip_event_create(ctypes.byref(event)) != 0:
        raise RuntimeError("cannot create an event")
    leaves = [Tensor(a, "hip", requires_grad=_trained(case, i), dtype=_dtype(case, i))
              for i, a in enumerate(_inputs(case, seed))]
    return {"case": dict(case), "in": leaves, "event": event}


# -------------------------------------------------------------------- pass --
class _Shared:
    """A realized tensor's buffer as torch sees it, without a copy; torch keeps
    this object, and so the buffer, as long as it uses the memory."""

    _TYPES = {"float32": "<f4", "int64": "<i8", "bfloat16": "<i2", "float16": "<f2"}

    def __init__(self, tensor):
        self.tensor = tensor
        self.__cuda_array_interface__ = {"shape": tensor.shape, "typestr": self._TYPES[tensor.dtype], "version": 2,
                                         "data": (tensor._node.data.ptr, False)}


def _hand_over(state, **tensors):
    """The realized tensors as torch tensors. Recording the event puts every
    launch that the library still holds back on the stream, where torch's own
    work follows it; it waits for none of them."""
    if _LIB.ormi_hip_event_record(state["event"]) != 0:
        raise RuntimeError("cannot record an event")
    out = {}
    for name, t in tensors.items():
        v = torch.as_tensor(_Shared(t), device="cuda")
        out[name] = v.view(torch.bfloat16) if t.dtype == "bfloat16" else v
    return out


def run(state):
    return _RUN[state["case"]["kind"]](state, *state["in"])


def _rows_train(state, a, b, c):
    for t in (a, b, c):
        t.zero_grad()
    y = ((a * b + c).relu() * 0.5).sum(1)
    loss = y.sum()
    loss.backward()
    ga, gb, gc = a.grad, b.grad, c.grad
    realize_all(y, ga, gb, gc)
    loss.zero_grad_graph()
    return _hand_over(state, y=y, ga=ga, gb=gb, gc=gc)


def _chain(state, x, bias, scale):
    z = ((x + bias) * scale).tanh() * x.sigmoid() - 0.1 * x * x
    if state["case"]["dtype"] != "float32":
        z = z.astype(state["case"]["dtype"])
    return _hand_over(state, z=z.realize())


def _stats(state, x):
    top = x.max(1, keepdims=True)
    denom = (x - top).exp().sum(1)
    mean, arg, cols = x.mean(1), x.argmax(1), x.sum(0)
    realize_all(top, denom, mean, arg, cols)
    return _hand_over(state, top=top, denom=denom, mean=mean, arg=arg, cols=cols)


def _norm(state, x, gamma, beta, dy):
    for t in (x, gamma, beta):
        t.zero_grad()
    centred = x - x.mean(1, keepdims=True)
    inv = ((centred * centred).mean(1, keepdims=True) + EPS) ** -0.5
    y = centred * inv * gamma + beta
    total = (y * dy).sum()
    total.backward()
    gx, ggamma, gbeta = x.grad, gamma.grad, beta.grad
    realize_all(y, gx, ggamma, gbeta)
    total.zero_grad_graph()
    return _hand_over(state, y=y, gx=gx, ggamma=ggamma, gbeta=gbeta)


def _swap(t):
    """The last two dims of a batch of matrices exchanged, as a view."""
    n = len(t.shape)
    return t.transpose(tuple(range(n - 2)) + (n - 1, n - 2))


def _gemm(state, a, b):
    layout = state["case"]["layout"]
    c = (_swap(a) if layout == "tn" else a) @ (_swap(b) if layout == "nt" else b)
    return _hand_over(state, c=c.realize())


def _gemm_grad(state, a, b, dc):
    a.zero_grad()
    b.zero_grad()
    c = a @ b
    total = (c * dc).sum()
    total.backward()
    ga, gb = a.grad, b.grad
    realize_all(c, ga, gb)
    total.zero_grad_graph()
    return _hand_over(state, c=c, ga=ga, gb=gb)


def _mlp_train(state, x, w0, w1, w2, target):
    ws = (w0, w1, w2)
    for w in ws:
        w.zero_grad()
    d = ((x @ w0).gelu() @ w1).gelu() @ w2 - target
    loss = (d * d).sum() * (1.0 / (target.shape[0] * target.shape[1]))
    loss.backward()
    new = [w - w.grad * LR for w in ws]
    realize_all(*new, loss)
    loss.zero_grad_graph()
    return _hand_over(state, w0=new[0], w1=new[1], w2=new[2], loss=loss)


def _mlp_infer(state, x, w0, w1, w2):
    h = (x @ w0).gelu().astype("bfloat16")
    h = (h @ w1).gelu().astype("bfloat16")
    return _hand_over(state, logits=(h @ w2).realize())


_RUN = {"rows_train": _rows_train, "chain": _chain, "stats": _stats, "norm": _norm, "gemm": _gemm,
        "gemm_grad": _gemm_grad, "mlp_train": _mlp_train, "mlp_infer": _mlp_infer}


# -------------------------------------------------------------------- work --
def work(case):
    """Bytes: each input read once, each output written once. Flops: the
    products' multiply-adds, and about one per element-wise operation."""
    kind = case["kind"]
    if kind in ("rows_train", "chain", "stats", "norm"):
        r, c = case["rows"], case["cols"]
        n = r * c
        if kind == "rows_train":
            return {"bytes": 24 * n + 4 * r, "flops": 10 * n}
        if kind == "chain":
            return {"bytes": 2 * n * (4 if case["dtype"] == "float32" else 2) + 4 * (r + c), "flops": 24 * n}
        if kind == "stats":
            return {"bytes": 4 * n + 20 * r + 4 * c, "flops": 12 * n}
        return {"bytes": 16 * n + 16 * c, "flops": 20 * n}
    if kind in ("gemm", "gemm_grad"):
        b, m, n, k = case.get("batch", 1), case["m"], case["n"], case["k"]
        if kind == "gemm":
            size = 4 if case["dtype"] == "float32" else 2
            return {"bytes": b * (size * (m * k + k * n) + 4 * m * n), "flops": 2 * b * m * n * k}
        return {"bytes": 4 * (2 * m * k + 2 * k * n + 2 * m * n), "flops": 6 * m * n * k}
    r, d = case["rows"], [case["d0"], case["d1"], case["d2"], case["d3"]]
    weights = sum(i * o for i, o in zip(d, d[1:]))
    if kind == "mlp_train":
        return {"bytes": 4 * (2 * weights + r * (d[0] + d[3])), "flops": 2 * r * (3 * weights - d[0] * d[1])}
    return {"bytes": 2 * (weights + r * d[0]) + 4 * r * d[3], "flops": 2 * r * weights}


# ------------------------------------------------------------------- exact --
def exact(case, seed):
    x = []
    for i, a in enumerate(_inputs(case, seed)):
        t = torch.from_numpy(a).cuda()
        x.append((t if _dtype(case, i) == "float32" else t.to(getattr(torch, _dtype(case, i)))).double())
    with torch.no_grad():
        return _EXACT[case["kind"]](case, *x)


def _exact_rows_train(case, a, b, c):
    z = a * b + c
    on = (z > 0).double() * 0.5
    return {"y": (z * on).sum(1), "ga": on * b, "gb": on * a, "gc": on}


def _exact_chain(case, x, bias, scale):
    return {"z": ((x + bias) * scale).tanh() * x.sigmoid() - 0.1 * x * x}


def _exact_stats(case, x):
    top, arg = x.max(1, keepdim=True)
    return {"top": top, "denom": (x - top).exp().sum(1), "mean": x.mean(1), "arg": arg[:, 0], "cols": x.sum(0)}


def _exact_norm(case, x, gamma, beta, dy):
    centred = x - x.mean(1, keepdim=True)
    inv = (centred.square().mean(1, keepdim=True) + EPS).rsqrt()
    unit = centred * inv
    g = dy * gamma
    gx = inv * (g - g.mean(1, keepdim=True) - unit * (g * unit).mean(1, keepdim=True))
    return {"y": unit * gamma + beta, "gx": gx, "ggamma": (dy * unit).sum(0), "gbeta": dy.sum(0)}


def _exact_gemm(case, a, b):
    a = a.transpose(-1, -2).contiguous() if case["layout"] == "tn" else a
    b = b.transpose(-1, -2).contiguous() if case["layout"] == "nt" else b
    return {"c": torch.stack([p @ q for p, q in zip(a, b)]) if a.dim() == 3 else a @ b}


def _exact_gemm_grad(case, a, b, dc):
    return {"c": a @ b, "ga": dc @ b.T, "gb": a.T @ dc}


def _gelu(z):
    return 0.5 * z * (1 + torch.erf(z * math.sqrt(0.5)))


def _gelu_grad(z):
    return 0.5 * (1 + torch.erf(z * math.sqrt(0.5))) + z * torch.exp(-0.5 * z * z) / math.sqrt(2 * math.pi)


def _exact_mlp_train(case, x, w0, w1, w2, target):
    z0 = x @ w0
    h0 = _gelu(z0)
    z1 = h0 @ w1
    h1 = _gelu(z1)
    d = h1 @ w2 - target
    scale = 1 / target.numel()
    dy = 2 * scale * d
    dz1 = (dy @ w2.T) * _gelu_grad(z1)
    dz0 = (dz1 @ w1.T) * _gelu_grad(z0)
    return {"w0": w0 - LR * (x.T @ dz0), "w1": w1 - LR * (h0.T @ dz1), "w2": w2 - LR * (h1.T @ dy),
            "loss": d.square().sum() * scale}


def _exact_mlp_infer(case, x, w0, w1, w2):
    return {"logits": _gelu(_gelu(x @ w0) @ w1) @ w2}


_EXACT = {"rows_train": _exact_rows_train, "chain": _exact_chain, "stats": _exact_stats, "norm": _exact_norm,
          "gemm": _exact_gemm, "gemm_grad": _exact_gemm_grad, "mlp_train": _exact_mlp_train, "mlp_infer": _exact_mlp_infer}


# --------------------------------------------------------------- tolerance --
def tolerance(case):
    """What another correct implementation at the same precision may differ by:
    float32 sums in another order, bfloat16 results one rounding apart."""
    kind = case["kind"]
    if kind == "chain":
        return {"rel": 2e-6 if case["dtype"] == "float32" else 4e-3}
    if kind == "mlp_infer":
        return {"rel": 1e-2}
    return {"rel": 1e-5}
