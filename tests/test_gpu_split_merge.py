"""Rows cut into chunks, in every transform-first aggregation and the sum form:
1 to 97 chunks a row (the merges take 2, 4 and 16 chunks' loads at a time), by
the default split of small graphs (128 edges) and by one of 64, and the static
layer at the edge of its scratch.

Transform-first rows are checked over the GPU's own Z, L and R as the row-group
test does: the row max bit for bit, den and output within 1e-5 of the sum of
magnitudes (FP32 sums of at most 1e4 terms, hardware exp2 at 2e-6 each; a
bf16-stored output adds 2^-8).  The sum form is compared with the oracle.
"""
import numpy as np
import pytest
import torch

import gatgpu
import oracle
from gatgpu import inputs
from test_gpu_row_groups import check_rows

pytestmark = pytest.mark.gpu

FINEST = {gatgpu.OPT_BLOCK_ROW_MIN_DEGREE: 0, gatgpu.OPT_SPLIT_ROW_MIN_DEGREE: 64, gatgpu.OPT_SPLIT_CHUNK_EDGES: 64}


def chunked_graph(n, chunk, counts, seed):
    """Rows of count * chunk - 1, count * chunk and count * chunk + 1 edges, the rest of 0 to 20."""
    rng = np.random.default_rng(seed)
    deg = rng.integers(0, 21, n)
    heavy = np.array([c * chunk + d for c in counts for d in (-1, 0, 1)])
    at = rng.choice(n, heavy.size, replace=False)
    deg[at] = heavy
    row = np.zeros(n + 1, np.uint64)
    np.cumsum(deg.astype(np.uint64), out=row[1:])
    return row, rng.integers(0, n, int(row[-1]), dtype=np.uint32), at


@pytest.fixture
def ctx():
    with gatgpu.Context(0) as c:  # options at their defaults, never set
        yield c


@pytest.mark.parametrize("K,d", [(8, 32), (8, 64), (1, 47), (4, 16), (6, 10), (3, 21)])
@pytest.mark.parametrize("precision", [gatgpu.FP32, gatgpu.BF16])
@pytest.mark.parametrize("chunk", [128, 64])
def test_chunk_counts(ctx, K, d, precision, chunk):
    n = 900
    row, col, heavy = chunked_graph(n, chunk, (1, 2, 3, 4, 5, 15, 16, 17, 33, 80 if chunk == 128 else 97), K * d)
    ctx.set_graph(row, col)
    if chunk == 64:
        for k, v in FINEST.items():
            ctx.set_option(k, v)
    ctx.set_layer(0, inputs.glorot_param(40, K, d, 6))
    for call in range(2):  # the arrival counters are left at zero
        x = inputs.normal((n, 40), 5 + call)
        ctx.set_input(x)
        ctx.layer_forward(0, precision, gatgpu.TRANSFORM_FIRST, call == 1)
        got = {k: ctx.stage(0, k) for k in ("left", "right", "max", "den", "out")}
        check_rows(ctx, row, col, K, d, got, call == 1, precision == gatgpu.BF16, np.concatenate([heavy, np.arange(40)]))


@pytest.mark.parametrize("d,din", [(32, 100), (64, 128)])
def test_chunk_counts_sum_form(ctx, d, din):
    n = 900
    row, col, _ = chunked_graph(n, 64, (1, 2, 3, 15, 16, 17, 97), d)
    p = inputs.glorot_param(din, 8, d, 6)
    ctx.set_graph(row, col)
    for k, v in FINEST.items():
        ctx.set_option(k, v)
    ctx.set_layer(0, p)
    qp = dict(p, w=oracle.quantize_bf16(p["w"]))
    for call in range(2):
        x = inputs.normal((n, din), 5 + call)
        ctx.set_input(x)
        ctx.layer_forward(0, gatgpu.BF16, gatgpu.AGGREGATE_FIRST, False)
        e = oracle.errors(oracle.ref_layer(row, col, oracle.quantize_bf16(x), qp, False)["out"], ctx.stage(0, "out"))
        assert e["finite"] and e["relative_l2"] < 1e-4, e


def test_static_layer_takes_the_coarse_split_at_the_limit(ctx):
    """8 x 64 bf16 on 25 700 nodes / 1.02M edges: 8 000 chunks of 128 edges need 17 MB and exceed the
    64 MiB array, where 512-edge rows in chunks of 256 fit as before."""
    n, rng = 25_700, np.random.default_rng(3)
    deg = rng.integers(1, 3, n)
    deg[:2100] = 460  # split into four chunks each by the fine split only
    row = np.zeros(n + 1, np.uint64)
    np.cumsum(deg.astype(np.uint64), out=row[1:])
    assert row[-1] < 1 << 20
    col = rng.integers(0, n, int(row[-1]), dtype=np.uint32)
    p = inputs.glorot_param(32, 8, 64, 6)
    x = inputs.normal((n, 32), 5)
    ctx.set_graph(row, col)
    ctx.set_layer(0, p)
    need = ctx.static_scratch_need(0, gatgpu.BF16, True)
    assert need <= gatgpu.STATIC_SCRATCH_BYTES
    xd = torch.from_numpy(x).cuda()
    od = torch.empty((n, 512), dtype=torch.float32, device="cuda")
    torch.cuda.synchronize()
    ctx.layer_forward_static(0, gatgpu.BF16, True, xd.data_ptr(), od.data_ptr())
    ctx.synchronize()
    e = oracle.errors(oracle.ref_layer(row, col, x, p, True)["out"], od.cpu().numpy())
    assert e["finite"] and e["relative_l2"] < 1e-2, e
    small = 20_000  # a graph whose fine split fits reports its larger need, still within the array
    ctx.set_graph(row[:small + 1], np.minimum(col[:int(row[small])], small - 1))
    assert ctx.static_scratch_need(0, gatgpu.BF16, True) <= gatgpu.STATIC_SCRATCH_BYTES


def test_options_set_and_restored(ctx):
    """Options 1 to 3 set and set back to their defaults: the split of a context that never set them
    (a graph below 1M edges cuts its rows of 128 edges on)."""
    row, col, _ = chunked_graph(900, 128, (1, 2, 3, 5, 17), 3)
    ctx.set_graph(row, col)
    ctx.set_layer(0, inputs.glorot_param(40, 8, 32, 6))
    need = lambda: ctx.static_scratch_need(0, gatgpu.BF16, True)
    fresh = need()
    for k, v, default in ((gatgpu.OPT_BLOCK_ROW_MIN_DEGREE, 600, 512), (gatgpu.OPT_SPLIT_ROW_MIN_DEGREE, 700, 0),
                          (gatgpu.OPT_SPLIT_CHUNK_EDGES, 512, 0)):
        ctx.set_option(k, v)
        assert need() < fresh  # fewer chunks
        ctx.set_option(k, default)
        assert need() == fresh
    ctx.set_option(gatgpu.OPT_BLOCK_ROW_MIN_DEGREE, 512)  # its default, before any other value
    assert need() == fresh


def test_static_need_per_chunk(ctx):
    """A chunk of a split row takes its partials (528 floats) and an arrival counter, and nothing else."""
    need = []
    for counts in ((), (1, 2, 3, 5, 17)):
        row, col, _ = chunked_graph(900, 128, counts, 3)
        ctx.set_graph(row, col)
        ctx.set_layer(0, inputs.glorot_param(40, 8, 32, 6))
        need.append(ctx.static_scratch_need(0, gatgpu.BF16, True))
    deg = np.diff(row.astype(np.int64))
    chunks = int(((deg[deg >= 128] + 127) // 128).sum())
    up = lambda b: (b + 255) // 256 * 256
    assert need[1] - need[0] == up(chunks * 528 * 4) + up(chunks * 4)
