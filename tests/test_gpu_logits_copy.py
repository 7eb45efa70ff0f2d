"""The ways logits leave gatgpu_model_forward: packed by a kernel into pinned
host memory (below 8 MB), packed and copied (more, or pageable or unaligned
memory), or as they are (rows without padding).  Every way gives the same bits.
"""
import numpy as np
import pytest
import torch

import gatgpu
from gatgpu import inputs

pytestmark = pytest.mark.gpu


def forward_into(ctx, precision, pointer):
    rc = ctx.lib.gatgpu_model_forward(ctx.h, precision, gatgpu.AUTO, pointer, None, None)
    assert rc == gatgpu.OK, ctx.lib.gatgpu_last_error(ctx.h)


# Below and above 8 MB; widths with and without padding; partial blocks of rows.
@pytest.mark.parametrize("n,edges,top,classes", [(1, 4, 0, 7), (1000, 9000, 300, 7), (32_767, 200_000, 900, 64),
                                                 (45_001, 400_003, 20_000, 47), (70_003, 500_000, 40, 33)])
@pytest.mark.parametrize("precision", [gatgpu.FP32, gatgpu.BF16])
def test_every_way_gives_the_same_rows(gpu_ctx, n, edges, top, classes, precision):
    ctx = gpu_ctx
    row, col = inputs.powerlaw_graph(n, edges, top, 5) if top else inputs.uniform_graph(n, edges, 5)
    ctx.set_graph(row, col)
    ctx.set_model(inputs.glorot_model(24, 8, 8, classes, 3))
    ctx.set_input(inputs.normal((n, 24), 4))
    want, _, _ = ctx.model_forward(precision, timed=True)
    assert np.all(np.isfinite(want)) and np.abs(want).max() > 0
    assert ctx.static_times()["logits_d2h_ms"] > 0
    got, _, _ = ctx.model_forward(precision, timed=False)
    assert np.array_equal(got, want), "pageable"
    assert ctx.static_times()["logits_d2h_ms"] > 0
    for offset in (0, 1):  # floats: the second start is not 16-byte aligned
        host = torch.full((n * classes + 8,), float("nan"), pin_memory=True)
        for _ in range(2):
            forward_into(ctx, precision, host.data_ptr() + 4 * offset)
        assert np.array_equal(host.numpy()[offset:offset + n * classes].reshape(n, classes), want), offset
        rest = np.concatenate([host.numpy()[:offset], host.numpy()[offset + n * classes:]])
        assert np.all(np.isnan(rest)), "wrote outside the logits"
    assert np.array_equal(ctx.stage(2, "out"), want)
