"""The row-group aggregation (csrc/aggregate.hip) at the edges of its dispatch:
every vector width, group size and vectors-per-lane count, rows of one batch
more or less, the change from a group to a wave per row, and split rows.

Checked over the GPU's own Z, L and R stages: the row max equals the scalar max
of LeakyReLU(L + R) bit for bit; den and the output equal a float64 softmax and
weighted sum.  Bounds: sums of at most 1e4 terms in FP32 with weights from the
hardware exp2 (2e-6 each), 1e-5 of the sum of magnitudes; a bf16-stored hidden
output adds half a bf16 ulp and the ELU error, 2^-8 relative.
"""
import numpy as np
import pytest

import gatgpu
from gatgpu import inputs

pytestmark = pytest.mark.gpu

# (K, d): groups of 8/16/32/64 lanes and 2/4/8 vectors a lane, in both types.
SHAPES = [(8, 8), (4, 16), (8, 16), (4, 64), (2, 64), (6, 12), (6, 10), (8, 60), (8, 46), (3, 21), (5, 33), (8, 63),
          (1, 1), (1, 5), (1, 32), (1, 47), (1, 60), (1, 61), (1, 64)]


def edge_graph(n, most, seed):
    """Rows of 0 to 70 edges each, then around every later edge of the dispatch."""
    rng = np.random.default_rng(seed)
    deg = np.concatenate([np.arange(71), [127, 128, 129, 255, 256, 257, 511, 512, 513, 1025, most], rng.integers(0, 12, n)])[:n]
    rng.shuffle(deg)
    row = np.zeros(n + 1, np.uint64)
    np.cumsum(deg.astype(np.uint64), out=row[1:])
    return row, rng.integers(0, n, int(row[-1]), dtype=np.uint32)


def check_rows(ctx, row, col, K, d, got, hidden, bf16, nodes):
    n = row.size - 1
    Z = ctx.stage(0, "z").astype(np.float64).reshape(n, K, d)
    L, R, M, den, out = (got[k] for k in ("left", "right", "max", "den", "out"))
    out = out.reshape(n, K, d)
    for i in nodes:
        b, e = int(row[i]), int(row[i + 1])
        if b == e:
            assert np.all(M[i] == 0) and np.all(den[i] == 0) and np.all(out[i] == 0), i
            continue
        src = col[b:e]
        s = L[i][None, :] + R[src]
        s = np.maximum(s, np.float32(0.2) * s)
        assert np.array_equal(s.max(axis=0), M[i]), (i, e - b)
        w = np.exp(s.astype(np.float64) - M[i].astype(np.float64))
        d64 = w.sum(axis=0)
        assert np.all(np.abs(den[i] - d64) <= 1e-5 * d64), (i, e - b)
        want = np.einsum("eh,ehf->hf", w, Z[src]) / d64[:, None]
        mag = np.einsum("eh,ehf->hf", w, np.abs(Z[src])) / d64[:, None]
        if hidden:
            want = np.where(want >= 0, want, np.expm1(want))
        tol = 1e-5 * mag + 1e-30 + (2.0 ** -8 * np.abs(want) if hidden and bf16 else 0)
        assert np.all(np.abs(out[i] - want) <= tol), (i, e - b)


@pytest.mark.parametrize("K,d", SHAPES)
@pytest.mark.parametrize("precision", [gatgpu.FP32, gatgpu.BF16])
def test_row_groups(gpu_ctx, K, d, precision):
    n = 700
    row, col = edge_graph(n, 1500, K * 64 + d)
    x = inputs.normal((n, 40), 5)
    p = inputs.glorot_param(40, K, d, 6)
    gpu_ctx.set_graph(row, col)
    gpu_ctx.set_layer(0, p)
    gpu_ctx.set_input(x)
    heaviest = np.argsort(np.diff(row.astype(np.int64)))
    nodes = np.unique(np.concatenate([heaviest[-90:], heaviest[:400:7]]))
    # default; every row of 16 edges or more cut into chunks of 64
    for options in ({}, {gatgpu.OPT_BLOCK_ROW_MIN_DEGREE: 16, gatgpu.OPT_SPLIT_ROW_MIN_DEGREE: 16,
                         gatgpu.OPT_SPLIT_CHUNK_EDGES: 64}):
        for k, v in options.items():
            gpu_ctx.set_option(k, v)
        try:
            for hidden in (False, True):
                gpu_ctx.layer_forward(0, precision, gatgpu.TRANSFORM_FIRST, hidden)
                got = {k: gpu_ctx.stage(0, k) for k in ("left", "right", "max", "den", "out")}
                check_rows(gpu_ctx, row, col, K, d, got, hidden, precision == gatgpu.BF16, nodes)
        finally:
            gpu_ctx.set_option(gatgpu.OPT_BLOCK_ROW_MIN_DEGREE, 512)
            gpu_ctx.set_option(gatgpu.OPT_SPLIT_ROW_MIN_DEGREE, 0)
            gpu_ctx.set_option(gatgpu.OPT_SPLIT_CHUNK_EDGES, 0)
