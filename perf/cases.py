"""Workloads of the sparse operators, called through the public entry points.

A case is one pass of something a graph-learning program does on the GPU: a neighbourhood sum
(``spmm_csr``, ``spmm_csr_auto``), its training step, a step on a freshly sampled mini-batch, edge
scores (``sddmm_csr_auto``), the softmax of edge scores over each node's edges, and graph attention
(``csr_attention_forward``).  The ranges:

* graphs of 1,000 to 1,000,000 nodes (plus the full 115M-edge skewed graph), 3 to 64 edges per node,
  with even degrees or a truncated power law whose columns prefer the nodes of high degree;
* feature widths from 8 to 256, among them class counts and raw input widths that are no multiple of
  the vector width;
* float32, bfloat16 and float16; with and without edge weights; forward, and forward + backward.

Graphs, features and weights are drawn on the GPU from the seed alone.  Schedules are decided, and
per-graph plans built, in ``prepare`` (one call), as a program does before its epochs; only the
mini-batch case meets a new graph in every pass.
"""

from __future__ import annotations

import math
import os
import tempfile

import torch

import autosage_amd
from autosage_amd.utils.csr import edge_index_to_csr

# The schedule cache is a file: a process decides for itself instead of replaying what another
# process (perhaps of another build) measured.
os.environ["AUTOSAGE_CACHE_DIR"] = tempfile.mkdtemp(prefix="autosage_cases_")

_DTYPES = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}
_CHUNK = 1 << 21


def _case(name, op, rows, degree, features, *, hub=0, value_features=0, dtype="f32", weighted=False, train=False):
    case = {"op": op, "rows": rows, "degree": degree, "hub": hub, "features": features,
            "value_features": value_features, "dtype": dtype, "weighted": weighted, "train": train}
    return case if name is None else {"name": name, **case}


def listed():
    return [
        # a citation-sized graph and a narrow hidden layer: the smallest calls, where latency counts
        _case("spmm small", "spmm", 3000, 4, 16, weighted=True),
        # one step of sampled training: edge_index -> CSR, sum, gradient; a new graph in every pass
        _case("minibatch step", "minibatch", 40000, 10, 100, train=True),
        # the last layer over a graph of 170k nodes with hubs: as many features as classes, an odd count
        _case("spmm classes", "spmm_auto", 170000, 14, 47, hub=10000, weighted=True),
        # 16 edges per node, one million nodes, F = 128, weighted: X is beyond every cache
        _case("spmm uniform 1M", "spmm", 1 << 20, 16, 128, weighted=True),
        # the benchmark's skewed graph: 233k nodes, 115M edges, hubs of up to 21,000 edges
        _case("spmm skewed 115M", "spmm_auto", 232965, 492, 128, hub=21000),
        # a training step with learned edge weights on raw input features (gradients of X and weights)
        _case("spmm train", "spmm", 200000, 16, 100, hub=1000, weighted=True, train=True),
        # 16-bit features of a wide hidden layer
        _case("spmm bf16", "spmm", 200000, 50, 256, hub=5000, dtype="bf16"),
        # edge scores on a hub-heavy graph, 16-bit
        _case("sddmm hubs f16", "sddmm", 500000, 40, 64, hub=100000, dtype="f16"),
        # edge scores between raw input features (no multiple of 32)
        _case("sddmm 100", "sddmm", 100000, 12, 100, hub=1000),
        # softmax over each node's edges and its gradient, as in additive graph attention
        _case("softmax train", "softmax", 1000000, 16, 1, hub=10000, train=True),
        # dot-product graph attention, one head, inference
        _case("attention", "attention", 600000, 30, 64, hub=10000, value_features=128),
        # dot-product graph attention, training in 16 bits
        _case("attention train bf16", "attention", 300000, 30, 64, hub=5000, value_features=64, dtype="bf16",
              train=True),
    ]


def _log_int(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    op = rng.choice(["spmm", "spmm_auto", "minibatch", "sddmm", "softmax", "attention"])
    rows = _log_int(rng, 1000, 1000000)
    degree = _log_int(rng, 3, 64)
    dtype = rng.choice(["f32", "f32", "bf16", "f16"])
    train = op == "minibatch" or rng.random() < 0.4

    def width():
        w = _log_int(rng, 8, 256)
        return w // 8 * 8 if rng.random() < 0.5 else w

    features, value_features = width(), 0
    hub = _log_int(rng, degree * 8, degree * 512) if rng.random() < 0.6 else 0
    if op == "minibatch":
        rows, hub = min(rows, 100000), 0
    if op == "softmax":
        features, dtype = 1, rng.choice(["f32", "f32", "f32", "bf16"])
    if op == "attention":
        value_features = width()
        if dtype != "f32":  # heads in 16 bits have widths that are multiples of 8
            features, value_features = (features + 7) // 8 * 8, (value_features + 7) // 8 * 8
    hub = min(hub, rows // 4)
    # a few milliseconds at most
    while rows * degree * (features + value_features) > 2_000_000_000:
        rows = rows * 2 // 3
    return _case(None, op, rows, degree, features, hub=hub, value_features=value_features, dtype=dtype,
                 weighted=op in ("spmm", "spmm_auto") and rng.random() < 0.5, train=train)


# ------------------------------------------------------------------------------------------------
# Graphs


def _row_pointers(case, gen):
    """Row pointers of a graph of rows x degree edges: even degrees (half to one and a half times the
    mean), or a power law of exponent 1.8 cut near ``hub`` and scaled to the mean."""
    n, mean, hub = case["rows"], case["degree"], case["hub"]
    if hub <= mean:
        real = torch.randint(mean - mean // 2, mean + mean // 2 + 1, (n,), generator=gen, device="cuda").double()
    else:
        raw = torch.rand(n, generator=gen, device="cuda", dtype=torch.float64).clamp_min_(1e-9).pow_(-1.25)
        low, high = 0.0, float(hub)
        for _ in range(40):
            middle = 0.5 * (low + high)
            if float((raw * middle).clamp_max_(hub).mean()) < mean:
                low = middle
            else:
                high = middle
        real = (raw * low).clamp_max_(hub)
    ends = real.cumsum(0)
    crow = torch.zeros(n + 1, dtype=torch.long, device="cuda")
    crow[1:] = (ends * (n * mean / ends[-1])).round().to(torch.long)
    return crow


def _graph(case, gen):
    """CSR with ascending columns.  Columns are uniform on even graphs, and drawn in proportion to
    the nodes' own degrees on power-law graphs."""
    n = case["rows"]
    crow = _row_pointers(case, gen)
    rows = _edge_rows(crow, n)
    if case["hub"] > case["degree"]:
        pick = torch.randint(0, rows.numel(), (rows.numel(),), generator=gen, device="cuda")
        columns = rows[pick]
        del pick
    else:
        columns = torch.randint(0, n, (rows.numel(),), generator=gen, device="cuda")
    keys = rows.mul_(n).add_(columns)
    del columns
    return crow, keys.sort().values.remainder_(n)


def _normal(shape, gen, dtype, scale=1.0):
    return (torch.randn(shape, generator=gen, device="cuda") * scale).to(dtype)


def prepare(case, seed):
    autosage_amd.load_native()
    gen = torch.Generator(device="cuda").manual_seed(seed)
    n, f, op = case["rows"], case["features"], case["op"]
    dtype = _DTYPES[case["dtype"]]
    state = {"case": case}
    if op == "minibatch":
        edges = n * case["degree"]
        state["edge_index"] = torch.randint(0, n, (2, edges), generator=gen, device="cuda")
        state["x"] = _normal((n, f), gen, dtype).requires_grad_(True)
        state["grad"] = _normal((n, f), gen, dtype)
        return state
    crow, col = _graph(case, gen)
    state["crow"], state["col"] = crow, col
    nnz = col.numel()
    train = case["train"]
    if op in ("spmm", "spmm_auto"):
        state["val"] = None
        if case["weighted"]:
            state["val"] = torch.rand(nnz, generator=gen, device="cuda").to(dtype).requires_grad_(train)
        state["x"] = _normal((n, f), gen, dtype).requires_grad_(train)
        out_width = f
    elif op in ("sddmm", "attention"):
        state["query"] = _normal((n, f), gen, dtype).requires_grad_(train)
        state["key"] = _normal((n, f), gen, dtype).requires_grad_(train)
        if op == "attention":
            out_width = case["value_features"]
            state["value"] = _normal((n, out_width), gen, dtype).requires_grad_(train)
            state["scale"] = 1.0 / math.sqrt(f)
    else:
        state["scores"] = _normal((nnz,), gen, dtype).requires_grad_(train)
    if train:
        state["grad"] = _normal((nnz,) if op in ("sddmm", "softmax") else (n, out_width), gen, dtype)
    run(state)  # schedules and plans
    return state


# ------------------------------------------------------------------------------------------------
# One pass


def run(state):
    case = state["case"]
    op = case["op"]
    if op == "minibatch":
        x = state["x"]
        crow, col = edge_index_to_csr(state["edge_index"], case["rows"])
        out = autosage_amd.spmm_csr(crow, col, None, x)
        (grad_x,) = torch.autograd.grad(out, (x,), state["grad"])
        return {"crow": crow, "col": col, "out": out.detach(), "grad_x": grad_x}
    crow, col = state["crow"], state["col"]
    if op == "spmm":
        names = ("x", "val")
        out = autosage_amd.spmm_csr(crow, col, state["val"], state["x"])
    elif op == "spmm_auto":
        names = ("x", "val")
        out, _ = autosage_amd.spmm_csr_auto(crow, col, state["val"], state["x"])
    elif op == "sddmm":
        names = ("query", "key")
        out, _ = autosage_amd.sddmm_csr_auto(crow, col, state["query"], state["key"])
    elif op == "softmax":
        names = ("scores",)
        out = torch.ops.autosage.csr_row_softmax(crow, state["scores"])
    else:
        names = ("query", "key", "value")
        out, _ = autosage_amd.csr_attention_forward(crow, col, state["query"], state["key"], state["value"],
                                                    scale=state["scale"])
    if not case["train"]:
        return {"out": out}
    names = [name for name in names if state[name] is not None]
    grads = torch.autograd.grad(out, [state[name] for name in names], state["grad"])
    return {"out": out.detach(), **{"grad_" + name: g for name, g in zip(names, grads)}}


# ------------------------------------------------------------------------------------------------
# What a pass cannot do without


def work(case):
    n, f, fv, op = case["rows"], case["features"], case["value_features"], case["op"]
    nnz = n * case["degree"]
    size = 4 if case["dtype"] == "f32" else 2
    index = 8 * nnz + 8 * (n + 1)
    train = case["train"]
    if op == "minibatch":
        # edge_index in, CSR out and read, X and dY in, Y and dX out
        return {"bytes": 16 * nnz + 2 * index + 4 * n * f * size, "flops": 4 * nnz * f}
    if op in ("spmm", "spmm_auto"):
        w = nnz * size if case["weighted"] else 0
        if not train:
            return {"bytes": index + w + 2 * n * f * size, "flops": 2 * nnz * f}
        # X, dY and the weights in; Y, dX and the weights' gradient out
        return {"bytes": index + 2 * w + 4 * n * f * size, "flops": (6 if case["weighted"] else 4) * nnz * f}
    if op == "sddmm":
        if not train:
            return {"bytes": index + 2 * n * f * size + nnz * size, "flops": 2 * nnz * f}
        return {"bytes": index + 4 * n * f * size + 2 * nnz * size, "flops": 6 * nnz * f}
    if op == "softmax":
        # scores in, probabilities out; with training also their gradient in and the scores' out
        return {"bytes": 8 * (n + 1) + (4 if train else 2) * nnz * size, "flops": (8 if train else 4) * nnz}
    dense = n * (2 * f + fv) * size + n * fv * size
    if not train:
        return {"bytes": index + dense, "flops": 2 * nnz * (f + fv)}
    return {"bytes": index + 2 * dense, "flops": 2 * nnz * (3 * f + 3 * fv) + 2 * nnz * f}


def tolerance(case):
    # About four times the distance from `exact`: 16-bit results are 1.7e-3 (bfloat16) and 2.1e-4
    # (float16) from it, one rounding of every value; float32 sums 4e-8 to 2e-7, and up to 3e-6 where
    # the rows of hubs are added up one edge after another.
    if case["dtype"] == "bf16":
        return {"rel": 7e-3}
    if case["dtype"] == "f16":
        return {"rel": 1e-3}
    return {"rel": 1e-5 if case["hub"] else 1e-6}


# ------------------------------------------------------------------------------------------------
# The same results in 64 bits, in plain torch


def _edge_rows(crow, n):
    return torch.repeat_interleave(torch.arange(n, device=crow.device), crow[1:] - crow[:-1])


def _product(crow, col, weights, x, n):
    """A·x in float64 for the CSR of the given weights."""
    return torch.sparse.mm(torch.sparse_csr_tensor(crow, col, weights, size=(n, n)), x)


def _transposed(crow, col, rows, n):
    order = col.argsort(stable=True)
    crow_t = torch.zeros_like(crow)
    crow_t[1:] = torch.bincount(col, minlength=n).cumsum(0)
    return crow_t, rows[order], order


def _dots(rows, col, a, b):
    out = torch.empty(rows.numel(), dtype=torch.float64, device=rows.device)
    for i in range(0, rows.numel(), _CHUNK):
        s = slice(i, i + _CHUNK)
        out[s] = (a[rows[s]] * b[col[s]]).sum(1)
    return out


def _row_sums(rows, values, n):
    return torch.zeros(n, dtype=torch.float64, device=rows.device).index_add_(0, rows, values)


def _softmax(rows, scores, n):
    top = torch.full((n,), -math.inf, dtype=torch.float64, device=rows.device)
    top.scatter_reduce_(0, rows, scores, reduce="amax")
    exps = (scores - top[rows]).exp()
    return exps / _row_sums(rows, exps, n)[rows]


def _softmax_grad(rows, probs, grad, n):
    return probs * (grad - _row_sums(rows, probs * grad, n)[rows])


def exact(case, seed):
    state = prepare(case, seed)
    n, op = case["rows"], case["op"]
    with torch.no_grad():
        wide = {k: v.detach().double() for k, v in state.items()
                if isinstance(v, torch.Tensor) and v.is_floating_point()}
        if op == "minibatch":
            src, dst = state["edge_index"]
            x, g = wide["x"], wide["grad"]
            out = torch.zeros_like(x).index_add_(0, dst, x[src])
            return {"crow": None, "col": None, "out": out, "grad_x": torch.zeros_like(x).index_add_(0, src, g[dst])}
        crow, col = state["crow"], state["col"]
        if op in ("spmm", "spmm_auto") and not case["train"]:
            weights = wide["val"] if case["weighted"] else torch.ones(col.numel(), dtype=torch.float64, device="cuda")
            return {"out": _product(crow, col, weights, wide["x"], n)}
        rows = _edge_rows(crow, n)
        if op == "softmax":
            probs = _softmax(rows, wide["scores"], n)
            if not case["train"]:
                return {"out": probs}
            return {"out": probs, "grad_scores": _softmax_grad(rows, probs, wide["grad"], n)}
        if op == "sddmm":
            out = _dots(rows, col, wide["query"], wide["key"])
            if not case["train"]:
                return {"out": out}
            crow_t, col_t, order = _transposed(crow, col, rows, n)
            return {"out": out, "grad_query": _product(crow, col, wide["grad"], wide["key"], n),
                    "grad_key": _product(crow_t, col_t, wide["grad"][order], wide["query"], n)}
        if op in ("spmm", "spmm_auto"):
            crow_t, col_t, order = _transposed(crow, col, rows, n)
            weights = wide["val"] if case["weighted"] else torch.ones(col.numel(), dtype=torch.float64, device="cuda")
            result = {"out": _product(crow, col, weights, wide["x"], n),
                      "grad_x": _product(crow_t, col_t, weights[order], wide["grad"], n)}
            if case["weighted"]:
                result["grad_val"] = _dots(rows, col, wide["grad"], wide["x"])
            return result
        query, key, value, scale = wide["query"], wide["key"], wide["value"], state["scale"]
        probs = _softmax(rows, _dots(rows, col, query, key) * scale, n)
        out = _product(crow, col, probs, value, n)
        if not case["train"]:
            return {"out": out}
        crow_t, col_t, order = _transposed(crow, col, rows, n)
        grad = wide["grad"]
        grad_s = _softmax_grad(rows, probs, _dots(rows, col, grad, value), n) * scale
        return {"out": out, "grad_query": _product(crow, col, grad_s, key, n),
                "grad_key": _product(crow_t, col_t, grad_s[order], query, n),
                "grad_value": _product(crow_t, col_t, probs[order], grad, n)}
