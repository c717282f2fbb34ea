"""PerRow activations on the matrix-core routes against exact sums of the oracle's codes: rows whose
scale is formed in the image launch and one block past them, token counts on both sides of that
launch's limit, of the batch and GEMM routes and of their tiles, a zero row, and an infinite and a
NaN value, which reach their own row only."""

import numpy as np
import pytest

from llmhost_amd import q4, synth

from .conftest import assert_close

pytestmark = pytest.mark.gpu


def _weights(blocks, n, k):
    b = blocks["qs"].reshape(n, k // 32, 16).astype(np.int64)
    nib = (np.stack([b & 15, b >> 4], axis=3).reshape(n, k // 32, 32) ^ 8) - 8
    return (nib * blocks["scale"].view(np.float16).astype(np.float64).reshape(n, -1, 1)).reshape(n, k)


@pytest.mark.parametrize("m,n,k", [(5, 40, 4096), (17, 33, 1568), (64, 64, 96), (9, 70, 4128), (65, 32, 4096),
                                   (97, 130, 1568), (70, 64, 4128), (128, 32, 2048), (129, 32, 2048)])
def test_row_image(gpu_ctx, oracle, m, n, k):
    blocks = synth.q4_blocks(n + k, n, k)
    x = synth.activations(m + k, m, k)
    x[1] = 0.0
    w = q4.Q4Matrix.from_blocks(n, k, blocks, gpu_ctx)
    y, z = (np.zeros((m, n), dtype=np.float32) for _ in range(2))
    q4.set_act_quant(q4.ActQuant.PerRow, gpu_ctx)
    try:
        q4.gemm_q4(w, x, y, m)
        xs = x.copy()
        xs[2, k - 1], xs[3, 0] = np.inf, np.nan
        q4.gemm_q4(w, xs, z, m)
    finally:
        q4.set_act_quant(q4.ActQuant.PerBlock, gpu_ctx)
        w.free()
    qs, sa, _ = oracle.act_quantize(x, True)
    a = qs.reshape(m, -1, 32).astype(np.float64) * sa.reshape(m, -1, 1).astype(np.float64)
    assert_close(y, a.reshape(m, k) @ _weights(blocks, n, k).T, what="per row")
    keep = ~np.isin(np.arange(m), (2, 3))
    assert np.array_equal(y[keep], z[keep])
