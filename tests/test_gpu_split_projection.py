"""The FP32 projection on split bf16 parts (csrc/projection_split.hip) at the
edges of its dispatch: input widths around whole k steps, one to three
launches, 1 to 16 output blocks (1, 2 or 4 tiles a block), L and R
shared between waves, inside a lane and by their own kernel, partial tiles.

Z, L and R against float64.  Bound: the split drops terms below 2^-25 of each
product and the rest is an FP32 sum, so an entry is within (D + 8) 2^-24 of the
sum of magnitudes (D additions of half an ulp each, and the dropped terms);
L and R add the width's additions over Z's own error.
"""
import numpy as np
import pytest

import gatgpu
from gatgpu import inputs

pytestmark = pytest.mark.gpu

SHAPES = [(1, 8, 32), (15, 1, 5), (16, 1, 47), (17, 2, 7), (33, 1, 64), (64, 4, 16), (65, 1, 32), (100, 8, 32),
          (112, 4, 32), (113, 3, 32), (128, 8, 64), (129, 7, 64), (200, 8, 63), (48, 8, 1), (70, 8, 2), (90, 5, 4), (256, 8, 32), (257, 8, 8), (300, 5, 33),
          (512, 2, 64), (513, 1, 40)]
EPS = 2.0 ** -24


def forward(ctx, n, D, K, d, x, p):
    row, col = inputs.uniform_graph(n, 4, 3)
    ctx.set_graph(row, col)
    ctx.set_layer(0, p)
    ctx.set_input(x)
    ctx.layer_forward(0, gatgpu.FP32, gatgpu.TRANSFORM_FIRST, False)
    return {k: ctx.stage(0, k) for k in ("z", "left", "right", "out")}


def check(got, x, p, K, d):
    n, D = x.shape
    x64, w64 = x.astype(np.float64), p["w"].astype(np.float64)
    z, mag = x64 @ w64, np.abs(x64) @ np.abs(w64)
    assert np.all(np.abs(got["z"] - z) <= (D + 8) * EPS * mag + 1e-37)
    for name, a in (("left", p["al"]), ("right", p["ar"])):
        a64 = a.astype(np.float64)
        dots = (z * a64).reshape(n, K, d).sum(axis=2)
        size = (mag * np.abs(a64)).reshape(n, K, d).sum(axis=2)
        assert np.all(np.abs(got[name] - dots) <= (D + d + 16) * EPS * size + 1e-37), name


@pytest.mark.parametrize("D,K,d", SHAPES)
@pytest.mark.parametrize("n", [1, 31, 97, 4099])
def test_split_projection(gpu_ctx, D, K, d, n):
    x = inputs.normal((n, D), D + n)
    p = inputs.glorot_param(D, K, d, 9)
    check(forward(gpu_ctx, n, D, K, d, x, p), x, p, K, d)


@pytest.mark.parametrize("D,K,d", [(100, 8, 32), (256, 1, 47), (300, 4, 16)])
def test_magnitudes_beyond_the_split(gpu_ctx, D, K, d):
    """Rows with inputs of 3.4e38 next to ordinary rows: the marked tiles take
    plain FP32 products, whose results stay finite where FP32's do."""
    n = 203
    x = inputs.normal((n, D), 4)
    p = inputs.glorot_param(D, K, d, 5)
    x[40, 3], x[199, D - 1] = np.float32(3.4028235e38), np.float32(-3.4e38)
    p["w"] *= np.float32(0.25)
    got = forward(gpu_ctx, n, D, K, d, x, p)
    assert np.all(np.isfinite(got["z"]))
    check({k: got[k] for k in ("z", "left", "right")}, x, p, K, d)


def test_weights_beyond_the_split(gpu_ctx):
    """A weight no bf16 holds: the layer keeps the VALU projection."""
    x = inputs.normal((65, 24), 4) * np.float32(1e-3)
    p = inputs.glorot_param(24, 2, 32, 5)
    p["w"][5, 7] = np.float32(3.4e38)
    p["al"][:] *= np.float32(1e-3)
    p["ar"][:] *= np.float32(1e-3)
    check(forward(gpu_ctx, 65, 24, 2, 32, x, p), x, p, 2, 32)
