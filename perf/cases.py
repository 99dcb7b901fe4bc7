"""Workloads of the tensor library, as its users run them.

Each case is one porch program over fp32 values that are already in HBM: a
fused elementwise chain, a view chain, softmaxes and row reductions, linear
layers forward and backward, products with one short side, an attention
layer, and a small classifier.  All but the classifier are driven as a
serving or training loop drives the library: the graph's node table is built
once, and a pass is one porch_materialize per result (include/porch_amd.h).
The classifier is written against the Python tensor API and records its
expression on every pass, as a short script does.

Results are the library's own device buffers, seen as torch tensors.
"""

from __future__ import annotations

import ctypes
import math

import torch

import porch_amd as porch
from porch_amd import _lib

# ---------------------------------------------------------------------------
# cases
# ---------------------------------------------------------------------------


def listed():
    return [
        # a two-layer classifier on a small batch: a few microseconds of
        # work in each kernel, so recording, planning and launches count
        {"name": "classifier", "kind": "classifier", "batch": 16, "features": 64, "hidden": 128,
         "classes": 10},
        # (a + b) * 2 - 1 over 2^20 values: one short fused launch
        {"name": "elementwise", "kind": "elementwise", "n": 1 << 20},
        # de-interleaving strided slices, transposed and joined: layout work
        {"name": "view_chain", "kind": "view_chain", "rows": 4096, "cols": 4096},
        # attention-sized and vocabulary-sized probability rows
        {"name": "softmax", "kind": "softmax", "rows": 8192, "cols": 4096},
        {"name": "vocab_softmax", "kind": "softmax", "rows": 512, "cols": 262144},
        # affine, relu, logistic and a sum per row: a pooled activation
        {"name": "logistic_rowsum", "kind": "rowsum", "rows": 16384, "cols": 2048},
        # a dense layer at a large, regular size
        {"name": "linear", "kind": "linear", "rows": 4096, "k": 4096, "cols": 4096, "wt": False},
        # a dense layer at sizes that divide no tile
        {"name": "linear_ragged", "kind": "linear", "rows": 777, "k": 1001, "cols": 3001,
         "wt": False},
        # the backward pass of a dense layer: the weight's, the input's and
        # the bias's gradients
        {"name": "linear_grads", "kind": "linear_grads", "rows": 4096, "k": 1024, "cols": 4096},
        # one token for each of 32 sequences against a weight: decoding
        {"name": "decode", "kind": "linear", "rows": 32, "k": 4096, "cols": 4096, "wt": False},
        # a matrix against a few columns: scoring heads, low-rank factors
        {"name": "narrow", "kind": "narrow", "rows": 4096, "k": 4096, "cols": 16},
        # softmax(q k^T / sqrt(d)) v over the heads of [batch, seq, heads, dim]
        # projections, back in [batch, seq, heads * dim]
        {"name": "attention", "kind": "attention", "batch": 2, "heads": 8, "seq": 4096, "dim": 64,
         "mask": False},
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _size(rng, lo, hi):
    """A size between lo and hi, even over its logarithm: any number (odd
    ones among them), a multiple of 8, or one of 128."""
    n = _log_int(rng, lo, hi)
    step = rng.choice((1, 1, 8, 128))
    return min(hi, max(lo, (n + step // 2) // step * step))


def draw(rng):
    kind = rng.choice(("classifier", "elementwise", "view_chain", "softmax", "rowsum", "linear",
                       "linear", "decode", "linear_grads", "narrow", "attention", "attention"))
    if kind == "classifier":
        return {"kind": kind, "batch": _size(rng, 1, 128), "features": _size(rng, 16, 512),
                "hidden": _size(rng, 32, 512), "classes": _size(rng, 2, 128)}
    if kind == "elementwise":
        return {"kind": kind, "n": _size(rng, 1000, 1 << 25)}
    if kind == "view_chain":
        # the slices take every second row and column: even extents
        return {"kind": kind, "rows": 2 * _size(rng, 64, 2048), "cols": 2 * _size(rng, 64, 2048)}
    if kind == "softmax":
        cols = _size(rng, 32, 1 << 18)
        return {"kind": kind, "cols": cols, "rows": _size(rng, 16, max(17, (1 << 26) // cols))}
    if kind == "rowsum":
        cols = _size(rng, 64, 16384)
        return {"kind": kind, "cols": cols, "rows": _size(rng, 64, (1 << 25) // cols)}
    if kind == "decode":
        return {"kind": "linear", "rows": _size(rng, 1, 64), "k": _size(rng, 512, 8192),
                "cols": _size(rng, 512, 8192), "wt": rng.random() < 0.5}
    if kind == "linear":
        return {"kind": kind, "rows": _size(rng, 64, 4096), "k": _size(rng, 128, 4096),
                "cols": _size(rng, 128, 4096), "wt": rng.random() < 0.5}
    if kind == "linear_grads":
        return {"kind": kind, "rows": _size(rng, 128, 4096), "k": _size(rng, 128, 2048),
                "cols": _size(rng, 128, 4096)}
    if kind == "narrow":
        return {"kind": kind, "rows": _size(rng, 256, 8192), "k": _size(rng, 256, 8192),
                "cols": rng.randint(1, 32)}
    batch, heads, dim = rng.choice((1, 2, 4)), rng.choice((4, 8, 12, 16)), rng.choice((32, 64, 128))
    # at most the listed case's products
    most = math.isqrt((2 * 8 * 4096 * 4096 * 64) // (batch * heads * dim))
    return {"kind": "attention", "batch": batch, "heads": heads, "seq": _size(rng, 64, min(4096, most)),
            "dim": dim, "mask": rng.random() < 0.5}


# ---------------------------------------------------------------------------
# inputs
# ---------------------------------------------------------------------------


def _values(case, seed):
    """The case's inputs as torch tensors on the GPU, in the graph's order."""
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)

    def normal(*shape, std=1.0, mean=0.0):
        return torch.randn(shape, generator=g, device="cuda") * std + mean

    def uniform(*shape, lo=-1.0, hi=1.0):
        return torch.rand(shape, generator=g, device="cuda") * (hi - lo) + lo

    kind = case["kind"]
    if kind == "classifier":
        f, h, c = case["features"], case["hidden"], case["classes"]
        return [normal(case["batch"], f), normal(f, h, std=f ** -0.5), normal(1, h, std=0.1),
                normal(h, c, std=h ** -0.5), normal(1, c, std=0.1)]
    if kind == "elementwise":
        return [uniform(case["n"]), uniform(case["n"])]
    if kind == "view_chain":
        return [normal(case["rows"], case["cols"])]
    if kind == "softmax":
        # a few dominant logits, as a trained model's rows have
        x = normal(case["rows"], case["cols"], std=3.0)
        return [torch.where(uniform(case["rows"], case["cols"], lo=0.0) < 0.01, 20.0, x)]
    if kind == "rowsum":
        n = case["cols"]
        return [normal(case["rows"], n), uniform(1, n, lo=0.5, hi=1.5), normal(1, n, std=0.1)]
    if kind == "linear":
        m, k, n = case["rows"], case["k"], case["cols"]
        w = (n, k) if case["wt"] else (k, n)
        return [normal(m, k), normal(*w, std=k ** -0.5), normal(1, n, std=0.1)]
    if kind == "linear_grads":
        m, k, n = case["rows"], case["k"], case["cols"]
        return [normal(m, k), normal(m, n, std=0.01), normal(k, n, std=k ** -0.5)]
    if kind == "narrow":
        m, k, n = case["rows"], case["k"], case["cols"]
        return [normal(m, k), normal(k, n, std=k ** -0.5)]
    if kind == "attention":
        shape = (case["batch"], case["seq"], case["heads"], case["dim"])
        values = [normal(*shape), normal(*shape), normal(*shape)]
        if case["mask"]:
            # causal, as an additive [seq, seq] tensor
            s = case["seq"]
            future = torch.ones((s, s), device="cuda", dtype=torch.bool).triu(1)
            values.append(torch.zeros((s, s), device="cuda").masked_fill_(future, -1e9))
        return values
    raise ValueError(kind)


# ---------------------------------------------------------------------------
# graphs
# ---------------------------------------------------------------------------


def _graphs(case, t):
    """The porch expressions of one pass over the tensors `t`."""
    kind = case["kind"]
    if kind == "classifier":
        x, w1, b1, w2, b2 = t
        m, h, c = case["batch"], case["hidden"], case["classes"]
        hidden = porch.relu(porch.matmul(x, w1) + porch.broadcast_to(b1, [m, h]))
        return [porch.softmax(porch.matmul(hidden, w2) + porch.broadcast_to(b2, [m, c]), 1)]
    if kind == "elementwise":
        a, b = t
        return [(a + b) * 2.0 - 1.0]
    if kind == "view_chain":
        (x,) = t
        r, c = case["rows"], case["cols"]
        return [porch.concat(porch.transpose(x[porch.slice(0, r, 2), porch.slice(1, c, 2)]),
                             porch.transpose(x[porch.slice(1, r, 2), porch.slice(0, c, 2)]), 0)
                + 1.0]
    if kind == "softmax":
        return [porch.softmax(t[0], 1)]
    if kind == "rowsum":
        x, w, b = t
        shape = [case["rows"], case["cols"]]
        return [porch.sum(porch.logistic(porch.relu(
            x * porch.broadcast_to(w, shape) + porch.broadcast_to(b, shape))), 1)]
    if kind == "linear":
        x, w, b = t
        product = porch.matmul(x, porch.transpose(w) if case["wt"] else w)
        return [porch.relu(product + porch.broadcast_to(b, [case["rows"], case["cols"]])) - 0.5]
    if kind == "linear_grads":
        x, dy, w = t
        return [porch.matmul(porch.transpose(x), dy), porch.matmul(dy, porch.transpose(w)),
                porch.sum(dy, 0)]
    if kind == "narrow":
        return [porch.matmul(t[0], t[1])]
    if kind == "attention":
        b, h, s, d = case["batch"], case["heads"], case["seq"], case["dim"]
        q, k, v = (porch.reshape(porch.permute(x, [0, 2, 1, 3]), [b * h, s, d]) for x in t[:3])
        scores = porch.batched_matmul(q, porch.permute(k, [0, 2, 1])) * (d ** -0.5)
        if case["mask"]:
            scores = scores + porch.broadcast_to(porch.unsqueeze(t[3], 0), [b * h, s, s])
        out = porch.reshape(porch.batched_matmul(porch.softmax(scores, 2), v), [b, h, s, d])
        return [porch.reshape(porch.permute(out, [0, 2, 1, 3]), [b, s, h * d])]
    raise ValueError(kind)


# ---------------------------------------------------------------------------
# device buffers as torch tensors, and passes over a kept node table
# ---------------------------------------------------------------------------


class _View:
    """A porch device buffer behind torch's array interface; torch keeps it,
    and the handle with it, for as long as a tensor reads the buffer."""

    def __init__(self, handle, shape, owns=True):
        self.handle = handle
        self.owner = owns
        self.__cuda_array_interface__ = {
            "shape": shape, "typestr": "<f4", "version": 2, "strides": None,
            "data": (_lib.lib.porch_buffer_device_pointer(handle), False)}

    def __del__(self):
        if self.owner:
            _lib.lib.porch_buffer_release(self.handle)


class _Pass:
    """One graph's node table and the handles of its inputs."""

    def __init__(self, expression):
        nodes, dims, n_dims, inputs, _ = porch.serialize(expression)
        self.graph = _lib.Graph(ctypes.cast(nodes, ctypes.POINTER(_lib.Node)), len(nodes),
                                ctypes.cast(dims, ctypes.POINTER(ctypes.c_int64)), n_dims)
        self.ref = ctypes.byref(self.graph)
        self.inputs = inputs
        self.handles = (ctypes.c_void_p * len(inputs))(*[t.device_data().handle for t in inputs])
        self.shape = tuple(expression.shape())
        self.out = ctypes.c_void_p()
        self.out_ref = ctypes.byref(self.out)

    def __call__(self):
        _lib.check(_lib.lib.porch_materialize(self.ref, self.handles, len(self.inputs),
                                              self.out_ref, None, 0, None))
        return torch.as_tensor(_View(self.out.value, self.shape), device="cuda")


def _device_tensor(values):
    """A porch tensor over its own device buffer, holding a torch tensor's values."""
    handle = ctypes.c_void_p()
    _lib.check(_lib.lib.porch_buffer_create(values.numel() * 4, ctypes.byref(handle)))
    _lib.check(_lib.lib.porch_synchronize())
    view = torch.as_tensor(_View(handle.value, tuple(values.shape), owns=False), device="cuda")
    view.copy_(values)
    return porch.tensor(porch.tensor_layout(values.shape), porch._Buffer(handle.value))


def prepare(case, seed):
    values = _values(case, seed)
    if case["kind"] == "classifier":
        return {"case": case, "tensors": [porch.tensor(list(v.shape), v.cpu().numpy())
                                          for v in values]}
    tensors = [_device_tensor(v) for v in values]
    torch.cuda.synchronize()  # the copies ran on torch's stream, porch reads on its own
    return {"case": case, "passes": [_Pass(e) for e in _graphs(case, tensors)]}


def run(state):
    if "tensors" in state:
        (expression,) = _graphs(state["case"], state["tensors"])
        y = porch.materialize(expression)
        view = _View(y.device_data().handle, y.shape(), owns=False)
        view.keep = y
        return torch.as_tensor(view, device="cuda")
    return [one() for one in state["passes"]]


# ---------------------------------------------------------------------------
# what a pass cannot do without, and how close a correct result is
# ---------------------------------------------------------------------------


def work(case):
    kind = case["kind"]
    if kind == "classifier":
        m, f, h, c = case["batch"], case["features"], case["hidden"], case["classes"]
        return {"bytes": 4 * (m * f + f * h + h + h * c + c + m * c),
                "flops": 2 * m * (f * h + h * c)}
    if kind == "elementwise":
        return {"bytes": 12 * case["n"], "flops": 3 * case["n"]}
    if kind == "view_chain":
        # half of x is kept, but every 128-byte line of it is read
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * n + 2 * n, "flops": n // 2}
    if kind == "softmax":
        n = case["rows"] * case["cols"]
        return {"bytes": 8 * n, "flops": 5 * n}
    if kind == "rowsum":
        n = case["rows"] * case["cols"]
        return {"bytes": 4 * (n + 2 * case["cols"] + case["rows"]), "flops": 7 * n}
    if kind in ("linear", "narrow"):
        m, k, n = case["rows"], case["k"], case["cols"]
        bias = n if kind == "linear" else 0
        return {"bytes": 4 * (m * k + k * n + bias + m * n), "flops": 2 * m * k * n}
    if kind == "linear_grads":
        m, k, n = case["rows"], case["k"], case["cols"]
        return {"bytes": 4 * (2 * m * k + m * n + 2 * k * n + n), "flops": 4 * m * k * n + m * n}
    b, h, s, d = case["batch"], case["heads"], case["seq"], case["dim"]
    return {"bytes": 4 * (4 * b * s * h * d + (s * s if case["mask"] else 0)),
            "flops": b * h * (4 * s * s * d + 5 * s * s)}


def tolerance(case):
    kind = case["kind"]
    if kind in ("elementwise", "view_chain"):
        return "exact"  # single IEEE operations in a given order
    if kind in ("softmax", "rowsum"):
        return {"rel": 1e-6, "max": 1e-5}  # exp within 2 ulp, 32-bit sums
    return {"rel": 1e-5, "max": 2e-4}  # 32-bit sums of products


def exact(case, seed):
    t = [v.double() for v in _values(case, seed)]
    kind = case["kind"]
    if kind == "classifier":
        x, w1, b1, w2, b2 = t
        return torch.softmax(torch.relu(x @ w1 + b1) @ w2 + b2, 1)
    if kind == "elementwise":
        return [(t[0] + t[1]) * 2.0 - 1.0]
    if kind == "view_chain":
        (x,) = t
        return [torch.cat([x[0::2, 1::2].T, x[1::2, 0::2].T], 0) + 1.0]
    if kind == "softmax":
        return [torch.softmax(t[0], 1)]
    if kind == "rowsum":
        return [torch.sigmoid(torch.relu(t[0] * t[1] + t[2])).sum(1)]
    if kind == "linear":
        x, w, b = t
        return [torch.relu(x @ (w.T if case["wt"] else w) + b) - 0.5]
    if kind == "linear_grads":
        x, dy, w = t
        return [x.T @ dy, dy @ w.T, dy.sum(0)]
    if kind == "narrow":
        return [t[0] @ t[1]]
    b, h, s, d = case["batch"], case["heads"], case["seq"], case["dim"]
    out = torch.empty((b, s, h, d), device="cuda", dtype=torch.float64)
    for i in range(b):
        for j in range(h):
            q, k, v = (x[i, :, j].contiguous() for x in t[:3])
            scores = (q @ k.T.contiguous()) * float(torch.tensor(d ** -0.5, dtype=torch.float32))
            if case["mask"]:
                scores += t[3]
            out[i, :, j] = torch.softmax(scores, 1) @ v
    return [out.reshape(b, s, h * d)]
