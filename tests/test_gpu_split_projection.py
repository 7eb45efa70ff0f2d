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
    """A weight no bf16 holds."""
    x = inputs.normal((65, 24), 4) * np.float32(1e-3)
    p = inputs.glorot_param(24, 2, 32, 5)
    p["w"][5, 7] = np.float32(3.4e38)
    p["al"][:] *= np.float32(1e-3)
    p["ar"][:] *= np.float32(1e-3)
    check(forward(gpu_ctx, 65, 24, 2, 32, x, p), x, p, 2, 32)


@pytest.mark.parametrize("D,K,d", [(24, 8, 8), (100, 8, 32), (256, 1, 47), (300, 4, 16), (70, 5, 33)])
@pytest.mark.parametrize("xs,ws", [(-118, 20), (-126, 60), (-140, 100), (20, -118), (60, -140), (0, -124), (-60, -60), (-100, -30), (-30, -70)])
def test_small_magnitudes(gpu_ctx, D, K, d, xs, ws):
    """Inputs or weights down to FP32's subnormals, scattered over 20 binades or all alike: every part
    of the split keeps its bits.  Bound: that of ordinary magnitudes, where each of the D + 8 roundings
    of a sum (D + d + 16 for the dots) is half a subnormal step, 2^-150, once the sum is below 2^-126."""
    n, rng = 97, np.random.default_rng(1000 + D + xs - ws)
    x = inputs.normal((n, D), 4)
    p = inputs.glorot_param(D, K, d, 5)
    x = np.ldexp(x, np.int64(xs) - rng.integers(0, 20, x.shape)).astype(np.float32)
    x[::2] = np.ldexp(inputs.normal((49, D), 6), xs).astype(np.float32)
    p["w"] = np.ldexp(p["w"], ws).astype(np.float32)
    got = forward(gpu_ctx, n, D, K, d, x, p)
    x64, w64 = x.astype(np.float64), p["w"].astype(np.float64)
    z, mag = x64 @ w64, np.abs(x64) @ np.abs(w64)
    step = 2.0 ** -150
    assert np.all(np.abs(got["z"] - z) <= (D + 8) * (EPS * mag + step))
    assert np.any(got["z"] != 0)
    for name, a in (("left", p["al"]), ("right", p["ar"])):
        a64 = a.astype(np.float64)
        dots = (z * a64).reshape(n, K, d).sum(axis=2)
        size = ((EPS * mag + step) * np.abs(a64)).reshape(n, K, d).sum(axis=2)
        assert np.all(np.abs(got[name] - dots) <= (D + d + 16) * (size + step)), name


def test_weights_of_every_magnitude(gpu_ctx):
    """A weight of 3.4e38 beside one of 1e-30: no factor keeps the parts of both."""
    x = inputs.normal((65, 24), 4) * np.float32(1e-3)
    p = inputs.glorot_param(24, 2, 32, 5)
    p["w"][5, 7], p["w"][6, 9], p["w"][3, 40] = np.float32(3.4e38), np.float32(1e-30), np.float32(-1e-40)
    p["al"][:] *= np.float32(1e-3)
    p["ar"][:] *= np.float32(1e-3)
    check(forward(gpu_ctx, 65, 24, 2, 32, x, p), x, p, 2, 32)


@pytest.mark.parametrize("D,K,d", [(40, 8, 32), (300, 1, 47), (40, 8, 8), (40, 3, 21)])
def test_products_beyond_fp32(gpu_ctx, D, K, d):
    """Finite operands whose product is not: infinite, with the sign, as FP32 products and sums are,
    and large finite results are themselves."""
    n = 97
    x = np.abs(inputs.normal((n, D), 4)) + np.float32(0.1)
    p = inputs.glorot_param(D, K, d, 5)
    sign = np.where(np.arange(K * d) % 2, np.float32(-1), np.float32(1))
    p["w"] = (np.abs(p["w"]) + np.float32(1e-3)) * np.float32(1e20) * sign
    p["al"][:] = p["ar"][:] = 0
    x[40] *= np.float32(1e25)   # beyond FP32
    x[41] *= np.float32(1e15)   # 1e35
    got = forward(gpu_ctx, n, D, K, d, x, p)["z"]
    assert np.all(got[40] == np.inf * sign)
    keep = np.arange(n) != 40
    z = x[keep].astype(np.float64) @ p["w"].astype(np.float64)
    assert np.all(np.abs(got[keep] - z) <= (D + 8) * EPS * np.abs(z))
