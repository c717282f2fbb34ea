"""A prompt's FFN block whose gate/up GEMM writes the down projection's operand image equals the
library's own op sequence bit for bit: token counts that end inside a 32-token tile and leave the
second token tile of a workgroup empty, an odd number of 32-row tiles of h (a padding block), odd
block counts of the model row, activations that overflow to inf, with and without the norm."""

import numpy as np
import pytest

from llmhost_amd import q4, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("norm", [True, False])
@pytest.mark.parametrize("dim,inter,tokens,big", [(64, 8192, 321, False), (1536, 8192, 97, False), (96, 8224, 350, False),
                                                  (1568, 10272, 260, False), (2048, 8192, 512, False),
                                                  (64, 8224, 385, True)])
def test_ffn_glu_equals_op_sequence(gpu_ctx, dim, inter, tokens, big, norm):
    shapes = ((inter, dim), (inter, dim), (dim, inter))
    w1, w3, w2 = (q4.Q4Matrix.from_blocks(n, k, synth.q4_blocks(80 + i + n, n, k), gpu_ctx)
                  for i, (n, k) in enumerate(shapes))
    x = synth.activations(81 + tokens, tokens, dim)
    x[3] = 0.0
    if big:  # g * u past f32: h holds inf, and NaN where silu(-inf) meets it
        x[5] *= np.float32(1e20)
    nw = (1 + 0.1 * synth.normal_f32(82, dim)).astype(np.float32) if norm else None
    got = x.copy()
    q4.ffn_residual(w1, w3, w2, nw, 1e-5, got, tokens)
    normed = x.copy()
    if norm:
        q4.rms_norm(x, nw, 1e-5, normed, gpu_ctx)
    g, u = (np.zeros((tokens, inter), dtype=np.float32) for _ in range(2))
    q4.norm_gemv([w1, w3], None, 1e-5, normed, [g, u], tokens)
    q4.silu_mul(g, u, gpu_ctx)
    ref = x.copy()
    q4.gemm_q4_add(w2, g, ref, tokens)
    for w in (w1, w3, w2):
        w.free()
    assert np.array_equal(got, ref, equal_nan=True)


def test_ffn_glu_long_rows(gpu_ctx):
    """Both sides of the rule for rows of 64 block pairs and more: 256 workgroups and more."""
    for dim, inter in ((4032, 8192), (4064, 8192), (4096, 8224)):
        test_ffn_glu_equals_op_sequence(gpu_ctx, dim, inter, 100, False, True)
