"""Two to four tokens over rows of 257 to 512 blocks (8 K slices in a workgroup) against the exact
value (64-bit sums of the oracle's codes), at the edges: one block past 8192 elements, the last row
length of 3 blocks per lane and one more, 16384 elements and one block past them (the matrix-core
route), rows that leave lanes idle, both act-quant modes and an addition."""

import numpy as np
import pytest

from llmhost_amd import q4, synth

from .conftest import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_row", [False, True])
@pytest.mark.parametrize("m,n,k", [(2, 33, 8224), (4, 70, 12288), (3, 64, 12320), (4, 5, 16384), (2, 130, 16416),
                                   (4, 2048, 10752)])
def test_batch_long_rows(gpu_ctx, oracle, m, n, k, per_row):
    blocks = synth.q4_blocks(n + k, n, k)
    x = synth.activations(m + k, m, k)
    y0 = synth.activations(m, m, n)
    w = q4.Q4Matrix.from_blocks(n, k, blocks, gpu_ctx)
    q4.set_act_quant(q4.ActQuant.PerRow if per_row else q4.ActQuant.PerBlock, gpu_ctx)
    try:
        got, added = np.zeros((m, n), dtype=np.float32), y0.copy()
        q4.gemm_q4(w, x, got, m)
        q4.gemm_q4_add(w, x, added, m)
    finally:
        q4.set_act_quant(q4.ActQuant.PerBlock, gpu_ctx)
        w.free()
    qs, sa, _ = oracle.act_quantize(x, per_row)
    wf = (synth_codes(blocks, n, k) * blocks["scale"].view(np.float16).astype(np.float64).reshape(n, -1, 1))
    a = qs.reshape(m, -1, 32).astype(np.float64) * sa.reshape(m, -1, 1).astype(np.float64)
    exact = a.reshape(m, k) @ wf.reshape(n, k).T
    assert_close(got, exact, what="gemm")
    assert_close(added, y0.astype(np.float64) + exact, what="gemm add")


def synth_codes(blocks, n, k):
    """Signed nibbles [n, k/32, 32] of BlockQ4 rows (element i in the low nibble of byte i/2 for even i)."""
    b = blocks["qs"].reshape(n, k // 32, 16).astype(np.int64)
    nib = np.stack([b & 15, b >> 4], axis=3).reshape(n, k // 32, 32)
    return (nib ^ 8) - 8
