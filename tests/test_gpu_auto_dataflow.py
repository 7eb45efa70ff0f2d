"""AUTO's dataflow of a bf16 layer depends on its Z table alone (the sum form above 256 MB), however
many edges the graph has: below the line model_forward and layer_forward both run transform-first,
with FP32 softmax weights and row sums, and carry its bits."""
import numpy as np
import pytest

import gatgpu
from gatgpu import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("din,dim,edges", [(40, 64, 1_600_000), (128, 64, 2_600_000), (100, 32, 6_100_000)])
def test_auto_below_the_z_line(din, dim, edges):
    n = 30_011
    row, col = inputs.powerlaw_graph(n, edges, 2000, 3)
    x = inputs.normal((n, din), 5)
    with gatgpu.Context(0) as ctx:
        ctx.set_graph(row, col)
        ctx.set_model(inputs.glorot_model(din, 8, dim, 7, 4))
        ctx.set_input(x)
        want, _, _ = ctx.model_forward(gatgpu.BF16, gatgpu.TRANSFORM_FIRST)
        stages = {k: ctx.stage(0, k) for k in ("z", "out", "left", "right", "max", "den")}
        got, _, _ = ctx.model_forward(gatgpu.BF16, gatgpu.AUTO)
        for k, v in stages.items():
            assert np.array_equal(ctx.stage(0, k), v), k
        assert np.array_equal(got, want)
        ctx.layer_forward(0, gatgpu.BF16, gatgpu.AUTO, True)
        assert np.array_equal(ctx.stage(0, "out"), stages["out"])
        # forced aggregate-first has no Z
        ctx.model_forward(gatgpu.BF16, gatgpu.AGGREGATE_FIRST)
        assert ctx.stage(0, "z") is None
