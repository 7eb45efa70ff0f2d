"""The one-block-a-wave projection (csrc/projection_tile.hip) at the edges of its
dispatch: 1 to 8 output blocks (4, 2 or 1 tiles a block), k steps of each
instantiation and around them, ragged input widths, partial tiles, more tiles
than blocks.  Z within one bf16 ulp and the FP32 ordering bound of the float64
product of the rounded operands, L within FP32 summation error of the dots, the
rounded rows (stage XBF) bit for bit; with 8 heads of 32, R within the error of
the dot of the GPU's own Z rows it is taken from.
"""
import numpy as np
import pytest
import torch

import gatgpu
import oracle
from gatgpu import inputs

pytestmark = pytest.mark.gpu

SHAPES = [(1, 1, 5), (16, 8, 4), (17, 1, 47), (64, 1, 61), (65, 4, 16), (100, 3, 32), (128, 8, 32), (129, 5, 32), (130, 8, 32),
          (200, 7, 28), (240, 8, 30), (256, 8, 32), (256, 1, 47), (257, 8, 8), (300, 2, 64), (500, 8, 8), (512, 7, 32),
          (512, 1, 16)]
EPS = 2.0 ** -24


@pytest.mark.parametrize("D,K,d", SHAPES)
@pytest.mark.parametrize("n", [1, 33, 1000, 20_011])
def test_tile_projection(gpu_ctx, D, K, d, n):
    x = inputs.normal((n, D), D + n)
    p = inputs.glorot_param(D, K, d, 9)
    row, col = inputs.uniform_graph(n, 4, 3)
    gpu_ctx.set_graph(row, col)
    gpu_ctx.set_layer(0, p)
    gpu_ctx.set_input(x)
    gpu_ctx.set_option(gatgpu.OPT_KEEP_INPUT_BF16, 1)
    try:
        gpu_ctx.layer_forward(0, gatgpu.BF16, gatgpu.TRANSFORM_FIRST, False)
        got = {k: gpu_ctx.stage(0, k) for k in ("z", "left", "right", "xbf")}
    finally:
        gpu_ctx.set_option(gatgpu.OPT_KEEP_INPUT_BF16, 0)
    xq, wq = oracle.quantize_bf16(x).astype(np.float64), oracle.quantize_bf16(p["w"]).astype(np.float64)
    assert np.array_equal(got["xbf"], oracle.quantize_bf16(x))
    z, mag = xq @ wq, np.abs(xq) @ np.abs(wq)
    ulp = np.ldexp(1.0, np.frexp(np.abs(z))[1] - 8)
    assert np.all(np.abs(got["z"] - z) <= ulp + 4 * D * EPS * mag)
    for name, a in (("left", p["al"]), ("right", p["ar"])):
        a64 = a.astype(np.float64)
        from_z = name == "right" and np.any([K == 8 and d == 32, K == 1 and d == 64])
        base = got["z"].astype(np.float64) if from_z and D <= 128 or from_z and 240 < D <= 256 else z
        terms, size = base * a64, mag * np.abs(a64)
        want = terms.reshape(n, K, d).sum(axis=2)
        # W a as bf16 hi + lo (2^-16 of it) and FP32 sums
        bound = (4 * (D + d) * EPS + 2.0 ** -16) * size.reshape(n, K, d).sum(axis=2)
        assert np.all(np.abs(got[name] - want) <= bound + 1e-30), name


@pytest.mark.parametrize("D,K,d,hidden", [(100, 8, 32, True), (33, 4, 16, True), (256, 1, 47, False), (64, 8, 64, True)])
def test_static_layer_unaligned_rows(gpu_ctx, D, K, d, hidden):
    """Device rows that start 4 bytes past 16-byte alignment: the same values
    as aligned ones, nothing written around them."""
    n, W = 1111, K * d
    row, col = inputs.powerlaw_graph(n, 20_000, 600, 3)
    gpu_ctx.set_graph(row, col)
    gpu_ctx.set_layer(0, inputs.glorot_param(D, K, d, 9))
    x = torch.from_numpy(inputs.normal((n, D), 4)).cuda()
    outs = []
    for shift in (0, 1):
        xs = torch.full((n * D + 4,), float("nan"), device="cuda")
        xs[shift:shift + n * D] = x.reshape(-1)
        out = torch.full((n * W + 4,), float("nan"), device="cuda")
        torch.cuda.synchronize()
        gpu_ctx.layer_forward_static(0, gatgpu.BF16, hidden, xs.data_ptr() + 4 * shift, out.data_ptr() + 4 * shift)
        gpu_ctx.synchronize()
        outs.append(out[shift:shift + n * W].cpu().numpy())
        assert torch.isnan(torch.cat([out[:shift], out[shift + n * W:]])).all()
    assert np.all(np.isfinite(outs[0])) and np.array_equal(outs[0], outs[1])


def check_r_in_rows(ctx, layer, col, n):
    """Rows of one edge each: the row max is LeakyReLU(L + R) of the R the aggregation reads in its
    source's Z row, so it carries that R's bits."""
    left, right, top = (ctx.stage(layer, k).reshape(n) for k in ("left", "right", "max"))
    s = left + right[col]
    assert np.array_equal(np.maximum(s, np.float32(0.2) * s), top)


@pytest.mark.parametrize("width", [1, 55, 56, 57, 58, 59, 60])
@pytest.mark.parametrize("D,n", [(40, 33), (256, 1000), (100, 20_011), (512, 20_011), (200, 70_001)])
def test_r_beside_the_last_features(gpu_ctx, width, D, n):
    """One head whose Z rows end in R: the widths whose last 16-byte piece of features holds it, and
    those just below, over partial tiles and 1 to 4 tiles a block."""
    row, col = np.arange(n + 1, dtype=np.uint64), ((np.arange(n) * 7 + 1) % n).astype(np.uint32)
    x = inputs.normal((n, D), D + n)
    p = inputs.glorot_param(D, 1, width, 9)
    gpu_ctx.set_graph(row, col)
    gpu_ctx.set_layer(0, p)
    gpu_ctx.set_input(x)
    gpu_ctx.layer_forward(0, gatgpu.BF16, gatgpu.TRANSFORM_FIRST, False)
    check_r_in_rows(gpu_ctx, 0, col, n)
    # one edge a row: the output is the source's Z row
    assert np.array_equal(gpu_ctx.stage(0, "out"), gpu_ctx.stage(0, "z")[col])


@pytest.mark.parametrize("classes", [57, 60])
def test_r_beside_the_last_features_from_bf16_rows(gpu_ctx, classes):
    """The same for the output layer of a model, whose input rows are bf16 already."""
    n = 20_011
    row, col = np.arange(n + 1, dtype=np.uint64), ((np.arange(n) * 7 + 1) % n).astype(np.uint32)
    gpu_ctx.set_graph(row, col)
    gpu_ctx.set_model(inputs.glorot_model(64, 8, 32, classes, 4))
    gpu_ctx.set_input(inputs.normal((n, 64), 5))
    logits, _, _ = gpu_ctx.model_forward(gatgpu.BF16, gatgpu.TRANSFORM_FIRST)
    check_r_in_rows(gpu_ctx, 2, col, n)
    assert np.array_equal(logits, gpu_ctx.stage(2, "z")[col])
