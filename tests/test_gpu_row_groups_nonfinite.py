"""The transform-first aggregations (csrc/aggregate.hip; -inf scores also csrc/aggregate_vec.hip) on
values that are not finite.

A batch's lanes past the row's last edge must not carry
another row's infinity or NaN into a row that is not connected to it; a row
connected to an infinite Z entry has that entry infinite, whatever the position
of the edge; and edges with a score of -inf weigh 0 as soon as the row has a
finite one, in whichever batch that comes.
"""
import numpy as np
import pytest
import torch

import gatgpu
from gatgpu import inputs
from test_gpu_row_groups import check_rows

pytestmark = pytest.mark.gpu

# (K, d) of the row-group kernel: 8, 16, 32 and 64 lanes, 2 and more vectors a lane; one head with R
# in the row, in its own array and recomputed from the row.
SHAPES = [(8, 8), (4, 16), (4, 64), (6, 10), (3, 21), (8, 46), (8, 63), (1, 5), (1, 47), (1, 61), (1, 64)]
# The default split, and every row of 16 edges or more cut into chunks of 64.
OPTIONS = [{}, {gatgpu.OPT_BLOCK_ROW_MIN_DEGREE: 16, gatgpu.OPT_SPLIT_ROW_MIN_DEGREE: 16,
                gatgpu.OPT_SPLIT_CHUNK_EDGES: 64}]


@pytest.fixture
def ctx():
    with gatgpu.Context(0) as c:
        yield c


def graph_of(rows):
    """CSR of the given neighbour lists."""
    row = np.zeros(len(rows) + 1, np.uint64)
    np.cumsum(np.array([len(r) for r in rows], np.uint64), out=row[1:])
    return row, np.concatenate([np.asarray(r, np.uint32) for r in rows])


def degrees(n, seed):
    deg = np.concatenate([np.arange(1, 71), [127, 128, 129, 255, 256, 257, 513], np.random.default_rng(seed).integers(1, 12, n)])[:n]
    return deg


@pytest.mark.parametrize("K,d", SHAPES)
@pytest.mark.parametrize("precision", [gatgpu.FP32, gatgpu.BF16])
@pytest.mark.parametrize("value", [float("nan"), float("inf")])
def test_unconnected_node_stays_apart(ctx, K, d, precision, value):
    """Node 0 has the fewest edges (so it is row 0 in degree order too) and no other node reads it."""
    n, D = 500, 24
    rng = np.random.default_rng(K * 64 + d)
    row, col = graph_of([[0]] + [rng.integers(1, n, k) for k in degrees(n - 1, 3) + 1])
    ctx.set_graph(row, col)
    ctx.set_layer(0, inputs.glorot_param(D, K, d, 6))
    x = torch.from_numpy(inputs.normal((n, D), 5)).cuda()
    out = torch.empty((n, K * d), device="cuda")
    for options in OPTIONS:
        for k, v in options.items():
            ctx.set_option(k, v)
        for hidden in (False, True):
            rows = []
            for first in (1.0, value):
                x[0] = first
                torch.cuda.synchronize()
                ctx.layer_forward_static(0, precision, hidden, x.data_ptr(), out.data_ptr())
                ctx.synchronize()
                rows.append(out.cpu().numpy())
            assert np.all(np.isfinite(rows[0]))
            assert not np.any(np.isfinite(rows[1][0]))
            # FP32 rows of the tile that holds node 0 may take the projection's other product:
            # another order of 24 additions in Z and the scores.
            tol = 0 if precision == gatgpu.BF16 else 2e-5 * np.abs(rows[0][1:]).max()
            assert np.all(np.abs(rows[1][1:] - rows[0][1:]) <= tol)


@pytest.mark.parametrize("K,d", [s for s in SHAPES if s != (1, 64)])  # (1, 64) takes R from the Z row
def test_infinite_feature_reaches_its_neighbours_only(ctx, K, d):
    """Z[j, 0] overflows while L and R of j stay finite (bf16: they are dots with W a, and a is 0
    there): feature 0 of a row is infinite where j is among its sources, first, last or between."""
    n, D = 400, 24
    rng = np.random.default_rng(K * 64 + d)
    deg = degrees(n - 1, 4) + 1
    rows = [[0]] + [rng.integers(2, n, k) for k in deg]
    hit = np.zeros(n, bool)
    for i in range(2, n, 3):
        rows[i][(0, -1, len(rows[i]) // 2)[(i // 3) % 3]] = 1
        hit[i] = True
    row, col = graph_of(rows)
    p = inputs.glorot_param(D, K, d, 6)
    p["w"][0, :] = 0
    p["w"][0, 0] = 16
    p["al"].reshape(-1)[0] = p["ar"].reshape(-1)[0] = 0
    x = inputs.normal((n, D), 5)
    x[:, 0] = 0
    x[1, 0] = np.float32(3e38)
    ctx.set_graph(row, col)
    ctx.set_layer(0, p)
    ctx.set_input(x)
    for options in OPTIONS:
        for k, v in options.items():
            ctx.set_option(k, v)
        ctx.layer_forward(0, gatgpu.BF16, gatgpu.TRANSFORM_FIRST, False)
        assert np.all(np.isfinite(ctx.stage(0, "right")))
        out = ctx.stage(0, "out")
        assert np.all(out[hit, 0] == np.inf)
        assert np.all(np.isfinite(out[~hit])) and np.all(np.isfinite(out[:, 1:]))


@pytest.mark.parametrize("K,d", SHAPES + [(8, 32), (8, 64)])
@pytest.mark.parametrize("precision", [gatgpu.FP32, gatgpu.BF16])
def test_scores_of_minus_infinity(ctx, K, d, precision):
    """R of some nodes overflows to -inf with Z and L finite; rows begin with 1 to 300 of them, or have
    them where a chunk of the row begins.  Rows of nothing else have no softmax: NaN, as
    exp(-inf - -inf) is."""
    n, D, low = 600, 24, 100  # nodes [0, low) have R = -inf
    rng = np.random.default_rng(K * 64 + d)
    rows = [[i % low if i < 40 else low + i] for i in range(200)]  # light rows of one edge
    for before in (1, 3, 4, 7, 8, 9, 16, 63, 64, 65, 128, 200, 300):
        for after in (0, 1, 4, 8, 40, 130):
            rows.append(np.concatenate([rng.integers(0, low, before), rng.integers(low, n, after)]))
    for lows in (1, 2, 16, 128, 150):
        for chunk in (64, 128, 256):
            rows.append(np.concatenate([rng.integers(low, n, chunk), rng.integers(0, low, lows), rng.integers(low, n, 200)]))
    rows += [rng.integers(0, n, k) for k in rng.integers(1, 30, n - len(rows))]
    row, col = graph_of(rows)
    p = inputs.glorot_param(D, K, d, 6)
    x = inputs.normal((n, D), 5)
    for h in range(K):  # one feature of each head is input h alone, and aR there is huge
        p["w"][h, :] = 0
        p["w"][:, h * d] = 0
        p["w"][h, h * d] = 1
        x[:, h] = 0
        x[:low, h] = -100
    p["al"].reshape(K, d)[:, 0] = 0
    p["ar"].reshape(K, d)[:, 0] = np.float32(3e38)
    ctx.set_graph(row, col)
    ctx.set_layer(0, p)
    ctx.set_input(x)
    none = np.array([np.all(np.asarray(r) < low) for r in rows])
    with np.errstate(invalid="ignore"):
        for options in OPTIONS:
            for k, v in options.items():
                ctx.set_option(k, v)
            for hidden in (False, True):
                ctx.layer_forward(0, precision, gatgpu.TRANSFORM_FIRST, hidden)
                got = {k: ctx.stage(0, k) for k in ("left", "right", "max", "den", "out")}
                assert np.all(got["right"][:low] == -np.inf) and np.all(np.isfinite(got["right"][low:]))
                assert np.all(np.isfinite(got["left"]))
                check_rows(ctx, row, col, K, d, got, hidden, precision == gatgpu.BF16, np.flatnonzero(~none))
                assert np.all(np.isnan(got["out"][none])) and np.all(np.isnan(got["den"][none]))
