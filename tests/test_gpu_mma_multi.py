"""Norm and projections of 2 to 4 tokens on both sides of the rule that norms in the kernel equal
rms_norm and one call per matrix.  Several matrices in one matrix-core batch launch (5 to 64 tokens) equal one launch each, bit for
bit: matrices of one plan, a matrix whose own plan differs (three token tiles past 8192 rows), rows
that end inside a 16-row tile, every number of token tiles, rows long enough for the form that loads
ahead (one and four token tiles)."""

import numpy as np
import pytest

from llmhost_amd import q4, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k,rows,tokens", [(2048, (2048, 512, 512), 40), (1568, (33, 1, 100), 5),
                                           (1536, (8200, 256, 8192), 37), (1536, (64, 8208, 8224), 48),
                                           (4096, (96, 130, 17), 64), (96, (48, 16), 17),
                                           (6176, (130, 33, 17), 9), (6176, (130, 33, 17), 53)])
def test_norm_gemv_equals_one_matrix_at_a_time(gpu_ctx, k, rows, tokens):
    ws = [q4.Q4Matrix.from_blocks(n, k, synth.q4_blocks(70 + i + n, n, k), gpu_ctx) for i, n in enumerate(rows)]
    x = synth.activations(71 + tokens, tokens, k)
    nw = (1 + 0.1 * synth.normal_f32(72, k)).astype(np.float32)
    outs = [np.full((tokens, n), np.nan, dtype=np.float32) for n in rows]
    q4.norm_gemv(ws, nw, 1e-5, x, outs, tokens)
    for w, got in zip(ws, outs):
        one = np.full_like(got, np.nan)
        q4.norm_gemv([w], nw, 1e-5, x, [one], tokens)
        assert np.array_equal(got.view(np.uint32), one.view(np.uint32))
    for w in ws:
        w.free()


@pytest.mark.parametrize("k,rows", [(512, (4096, 4096)), (512, (8192, 1)), (992, (8224,)), (1024, (8192, 8192)),
                                    (1024, (16385,)), (2048, (300, 32768, 17)), (64, (33000,))])
@pytest.mark.parametrize("tokens", [2, 3, 4])
def test_norm_gemv_few_tokens_equals_op_sequence(gpu_ctx, k, rows, tokens):
    ws = [q4.Q4Matrix.from_blocks(n, k, synth.q4_blocks(80 + i + n, n, k), gpu_ctx) for i, n in enumerate(rows)]
    x = synth.activations(81 + tokens, tokens, k)
    nw = (1 + 0.1 * synth.normal_f32(82, k)).astype(np.float32)
    outs = [np.full((tokens, n), np.nan, dtype=np.float32) for n in rows]
    q4.norm_gemv(ws, nw, 1e-5, x, outs, tokens)
    normed = np.empty_like(x)
    q4.rms_norm(x, nw, 1e-5, normed, gpu_ctx)
    for w, got in zip(ws, outs):
        one = np.full_like(got, np.nan)
        q4.gemm_q4(w, normed, one, tokens)
        assert np.array_equal(got.view(np.uint32), one.view(np.uint32))
        w.free()
