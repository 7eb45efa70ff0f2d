"""AUTO's edge rule for the model's first layer (sum form from 1.5M edges with 8 heads of 64): the
logits stay within the bf16 bound of transform-first, stage Z is still there and
carries transform-first's bits, and below the line nothing changes."""
import numpy as np
import pytest

import gatgpu
from gatgpu import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("din,edges,sums", [(40, 1_499_999, False), (40, 1_500_000, True), (100, 1_700_003, True),
                                            (128, 2_400_001, False), (128, 2_600_000, True), (13, 1_600_000, True)])
def test_sum_form_from_edges(din, edges, sums):
    n = 30_011
    row, col = inputs.powerlaw_graph(n, edges, 2000, 3)
    edges = int(row[-1])
    x = inputs.normal((n, din), 5)
    with gatgpu.Context(0) as ctx:
        ctx.set_graph(row, col)
        ctx.set_model(inputs.glorot_model(din, 8, 64, 7, 4))
        ctx.set_input(x)
        want, _, _ = ctx.model_forward(gatgpu.BF16, gatgpu.TRANSFORM_FIRST)
        stages = {k: ctx.stage(0, k) for k in ("z", "out", "left", "right", "max", "den")}
        for _ in range(2):
            got, _, _ = ctx.model_forward(gatgpu.BF16, gatgpu.AUTO)
            assert np.array_equal(got, want) == (not sums)
            before = {k: ctx.stage(0, k) for k in stages if k != "z"}
            assert np.array_equal(ctx.stage(0, "z"), stages["z"])
            for k, v in before.items():  # asking for Z leaves the other stages alone
                assert np.array_equal(ctx.stage(0, k), v)
                # two correct bf16 roundings of one result
                assert np.linalg.norm(v - stages[k]) <= 1.2e-2 * np.linalg.norm(stages[k]), k
            assert np.linalg.norm(got - want) <= 1.2e-2 * np.linalg.norm(want)
        # forced aggregate-first has no Z, as before
        ctx.model_forward(gatgpu.BF16, gatgpu.AGGREGATE_FIRST)
        assert ctx.stage(0, "z") is None
