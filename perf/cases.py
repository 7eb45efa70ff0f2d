"""The work a user of this framework has it do, as measurable cases.

Two entry points carry the cases:

* ``gatgpu_model_forward`` (C ABI): the three-layer forward
  ``D -> K x d -> K x d -> 1 x C`` over a resident graph, its logits copied to
  a host buffer the caller owns.  The buffer is pinned, as a serving program
  keeps it.
* ``layer_forward_static``: one layer on device-resident rows, no allocation.
  The scratch array behind it is shared by every context of a GPU, so a
  program that holds several contexts waits for one call before the next.

A case names its graph family (``uniform``, ``powerlaw``: in-degrees follow a
power law, ``rmat``: R-MAT, in- and out-degrees skewed, many rows with the
self-loop alone), its sizes, the layer shapes and the precision.  Every graph
has one self-loop per node, as the framework's generators make them.
"""
import math
import os
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.getcwd(), "gat-tfs_amd"))
import gatgpu  # noqa: E402
from gatgpu import inputs  # noqa: E402

PRECISION = {"fp32": gatgpu.FP32, "bf16": gatgpu.BF16}
STATIC_BYTES = gatgpu.STATIC_SCRATCH_BYTES


def _model(name, graph, n, edges, max_degree, din, heads, dim, classes, precision):
    return {"name": name, "entry": "model", "graph": graph, "n": n, "edges": edges, "max_degree": max_degree,
            "din": din, "heads": heads, "dim": dim, "classes": classes, "precision": precision}


def _layer(name, graph, n, edges, max_degree, din, heads, dim, hidden, precision):
    return {"name": name, "entry": "layer", "graph": graph, "n": n, "edges": edges, "max_degree": max_degree,
            "din": din, "heads": heads, "dim": dim, "hidden": hidden, "precision": precision}


def listed():
    return [
        # Smallest calls: one layer, and the whole model, on the 1024-node smoke graph.  A
        # latency-bound request, e.g. inference on a sampled neighbourhood.
        _layer("layer_1k_bf16", "uniform", 1024, 1024 * 16, 0, 128, 8, 32, True, "bf16"),
        _model("model_1k_bf16", "uniform", 1024, 1024 * 16, 0, 128, 8, 32, 40, "bf16"),
        # One hidden layer and one output layer of the same model inside a program that keeps its
        # rows on the GPU: ragged node counts, power-law in-degrees.
        _layer("layer_30k_hidden_bf16", "powerlaw", 30011, 450_037, 2500, 256, 8, 32, True, "bf16"),
        _layer("layer_60k_output_bf16", "powerlaw", 60013, 1_200_011, 4000, 256, 1, 47, False, "bf16"),
        # A narrower hidden layer (4 heads of 16) in FP32.
        _layer("layer_20k_4x16_fp32", "powerlaw", 20021, 300_007, 1500, 64, 4, 16, True, "fp32"),
        # A small citation-style graph: wide input features, 8 heads of 8, few classes.
        _model("model_20k_8x8_bf16", "powerlaw", 20011, 160_009, 170, 500, 8, 8, 7, "bf16"),
        # The 2.5M-edge graph of the published baseline, in both precisions.
        _model("model_2m5_bf16", "powerlaw", 169_343, 2_484_941, 13_162, 128, 8, 32, 40, "bf16"),
        _model("model_2m5_fp32", "powerlaw", 169_343, 2_484_941, 13_162, 128, 8, 32, 40, "fp32"),
        # Input widths that are not a power of two: 100 features, FP32 and bf16, between the 2.5M-
        # and the 64.3M-edge graph.
        _model("model_1m5_d100_fp32", "powerlaw", 120_011, 1_500_007, 8000, 100, 8, 32, 47, "fp32"),
        _model("model_9m_d100_bf16", "powerlaw", 360_007, 9_000_011, 12_000, 100, 8, 32, 47, "bf16"),
        # R-MAT skew with heads of 64 (the skew workload's layers, a quarter of its graph).
        _model("model_rmat_8x64_bf16", "rmat", 1 << 20, 24_000_000, 0, 128, 8, 64, 16, "bf16"),
        # The headline workload: 64.3M edges.
        _model("model_64m_bf16", "powerlaw", 2_449_029, 64_300_000, 17_000, 100, 8, 32, 47, "bf16"),
    ]


HIDDEN = [(8, 32), (8, 32), (8, 32), (8, 64), (4, 32), (4, 16), (8, 8), (8, 16), (2, 64), (4, 64), (1, 64), (6, 10)]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _graph(rng, n_lo, n_hi, edges_hi):
    """A graph family and sizes: (family, n, edges, max in-degree)."""
    n = _log_int(rng, n_lo, n_hi)
    degree = math.exp(rng.uniform(math.log(4), math.log(60)))
    edges = min(int(n * degree), edges_hi)
    family = rng.choice(("powerlaw", "powerlaw", "uniform", "rmat"))
    if family == "rmat":
        scale = max(10, min(20, n.bit_length() - 1))
        return family, 1 << scale, min(edges, 20 << scale), 0
    if family == "uniform":
        return family, n, n * max(2, int(edges / n)), 0
    cap = int(max(40 * edges / n, min(n / 8, 16_000)))
    return family, n, edges, max(2, min(cap, n - 1))


def draw(rng):
    precision = rng.choice(("bf16", "bf16", "fp32"))
    heads, dim = rng.choice(HIDDEN)
    if rng.random() < 0.4:  # one layer on device rows
        hidden = rng.random() < 0.6
        if not hidden:
            heads, dim = 1, rng.randint(2, 64)
        din = _log_int(rng, 16, 300)
        # rows: rounded input, Z, output and four softmax arrays; split rows: 2.2 KB per 256 edges
        row_bytes = 2 * (din + 16) + 8 * (heads * dim + 64) + 16 * heads
        n_hi = min(80_000, (STATIC_BYTES * 3 // 4) // row_bytes)
        family, n, edges, cap = _graph(rng, 600, n_hi, 1_200_000)
        if family == "rmat" and n > n_hi:
            n, edges = n // 2, edges // 2
        return {"entry": "layer", "graph": family, "n": n, "edges": edges, "max_degree": cap, "din": din,
                "heads": heads, "dim": dim, "hidden": hidden, "precision": precision}
    family, n, edges, cap = _graph(rng, 800, 700_000, 16_000_000 if precision == "bf16" else 8_000_000)
    return {"entry": "model", "graph": family, "n": n, "edges": edges, "max_degree": cap,
            "din": _log_int(rng, 16, 512), "heads": heads, "dim": dim, "classes": rng.randint(2, 64),
            "precision": precision}


def _rmat(scale, edges, seed):
    """R-MAT (0.57, 0.19, 0.19, 0.05): `edges` drawn edges and a self-loop per node, duplicates dropped."""
    g = torch.Generator(device="cuda").manual_seed(seed)
    dst = torch.zeros(edges, dtype=torch.int64, device="cuda")
    src = torch.zeros(edges, dtype=torch.int64, device="cuda")
    for _ in range(scale):
        u = torch.rand(edges, generator=g, device="cuda")
        dst = dst * 2 + (u >= 0.76)
        src = src * 2 + (((u >= 0.57) & (u < 0.76)) | (u >= 0.95))
    n = 1 << scale
    loops = torch.arange(n, device="cuda")
    keys = torch.unique(torch.cat([dst * n + src, loops * n + loops]))
    row = torch.zeros(n + 1, dtype=torch.int64, device="cuda")
    row[1:] = torch.cumsum(torch.bincount(keys // n, minlength=n), 0)
    return row.cpu().numpy().astype(np.uint64), (keys % n).cpu().numpy().astype(np.uint32)


def _graph_of(case, seed):
    n, edges = case["n"], case["edges"]
    if case["graph"] == "rmat":
        return _rmat(n.bit_length() - 1, edges, seed)
    if case["graph"] == "uniform":
        return inputs.uniform_graph(n, edges // n, seed)
    return inputs.powerlaw_graph(n, edges, case["max_degree"], seed)


def _inputs(case, seed):
    """Graph and weights on the host, N(0, 1) features on the GPU."""
    row, col = _graph_of(case, seed)
    g = torch.Generator(device="cuda").manual_seed(seed + 1)
    x = torch.randn(row.size - 1, case["din"], generator=g, device="cuda")
    if case["entry"] == "layer":
        params = [inputs.glorot_param(case["din"], case["heads"], case["dim"], seed + 2)]
    else:
        params = inputs.glorot_model(case["din"], case["heads"], case["dim"], case["classes"], seed + 2)
    return row, col, x, params


def prepare(case, seed):
    row, col, x, params = _inputs(case, seed)
    ctx = gatgpu.Context(0)
    ctx.set_graph(row, col)
    state = {"case": case, "ctx": ctx, "precision": PRECISION[case["precision"]]}
    if case["entry"] == "layer":
        ctx.set_layer(0, params[0])
        state["x"] = x
        state["out"] = torch.empty(x.shape[0], case["heads"] * case["dim"], device="cuda")
    else:
        ctx.set_model(params)
        ctx.set_input(x.cpu().numpy())
        state["logits"] = torch.empty(x.shape[0], case["classes"], pin_memory=True)
    return state


def run(state):
    ctx = state["ctx"]
    if state["case"]["entry"] == "layer":
        ctx.layer_forward_static(0, state["precision"], state["case"]["hidden"], state["x"].data_ptr(),
                                 state["out"].data_ptr())
        ctx.synchronize()
        return state["out"]
    rc = ctx.lib.gatgpu_model_forward(ctx.h, state["precision"], gatgpu.AUTO, state["logits"].data_ptr(), None, None)
    if rc != gatgpu.OK:
        raise gatgpu.GatGpuError(rc, ctx.lib.gatgpu_last_error(ctx.h).decode())
    return state["logits"]


def _shapes(case):
    if case["entry"] == "layer":
        return [(case["din"], case["heads"], case["dim"])]
    return inputs.model_dims(case["din"], case["heads"], case["dim"], case["classes"])


def work(case):
    """Features, CSR and weights read once, the last output written once; the products of the
    projections, the attention dots and, per edge and head, the score and the weighted sum."""
    n, e, shapes = case["n"], case["edges"], _shapes(case)
    nbytes = 4 * n * case["din"] + 8 * (n + 1) + 4 * e + 4 * n * shapes[-1][1] * shapes[-1][2]
    flops = 0
    for din, heads, dim in shapes:
        w = heads * dim
        nbytes += 4 * (din * w + 2 * w)
        flops += 2 * n * din * w + 4 * n * w + e * (6 * heads + 2 * w)
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    # bf16 inputs, weights and Z rows (2^-9 each, averaged over a row's edges): 3.1e-3 to 4.9e-3 off
    # the 64-bit result, and another correct rounding as far from it on its own side.  FP32: 1.9e-7
    # to 3.1e-7 off it, four times that for sums in another order.
    return {"rel": 1.2e-2} if case["precision"] == "bf16" else {"rel": 1.2e-6}


def _exact_layer(row, dst, src, h, p, hidden):
    """One layer in 64 bits: softmax over each destination's edges, weighted sum of Z rows, ELU."""
    n, heads, dim = row.numel() - 1, p["heads"], p["dim"]
    w, al, ar = (torch.from_numpy(p[k]).cuda().double() for k in ("w", "al", "ar"))
    z = (h @ w).view(n, heads, dim)
    left, right = (z * al.view(1, heads, dim)).sum(-1), (z * ar.view(1, heads, dim)).sum(-1)
    score = torch.nn.functional.leaky_relu(left[dst] + right[src], 0.2)
    top = torch.full((n, heads), -math.inf, dtype=torch.float64, device="cuda")
    top.scatter_reduce_(0, dst.view(-1, 1).expand(-1, heads), score, "amax")
    weight = torch.exp(score - top[dst])
    den = torch.zeros((n, heads), dtype=torch.float64, device="cuda").index_add_(0, dst, weight)
    out = torch.zeros((n, heads, dim), dtype=torch.float64, device="cuda")
    step = max(1, (1 << 27) // (heads * dim))
    for at in range(0, src.numel(), step):
        part = slice(at, at + step)
        out.index_add_(0, dst[part], weight[part].unsqueeze(-1) * z[src[part]])
    out = (out / den.unsqueeze(-1)).reshape(n, heads * dim)  # every node has its self-loop
    return torch.nn.functional.elu(out) if hidden else out


def exact(case, seed):
    row, col, x, params = _inputs(case, seed)
    row = torch.from_numpy(row.astype(np.int64)).cuda()
    src = torch.from_numpy(col.astype(np.int64)).cuda()
    dst = torch.repeat_interleave(torch.arange(row.numel() - 1, device="cuda"), row[1:] - row[:-1])
    h = x.double()
    if case["entry"] == "layer":
        return _exact_layer(row, dst, src, h, params[0], case["hidden"])
    for l, p in enumerate(params):
        h = _exact_layer(row, dst, src, h, p, l < 2)
    return h
