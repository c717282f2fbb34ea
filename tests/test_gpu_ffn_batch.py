"""The FFN block of 2 to 32 tokens (two or three fused launches) equals the library's own op sequence bit for
bit: every token slot count, rows that end inside a block group, a down projection whose kernel
takes codes (inter 2080-8192), f32 rows (shorter) or the matrix-core batch route (longer); from 5
tokens on, one and two token tiles, block counts of h that pad its image's quad by 0 to 3, rows of
33 to 65 blocks and one more slice chunk, and on both sides of the longest that are fused; both act-quant
modes, with and without the norm."""

import numpy as np
import pytest

from llmhost_amd import q4, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("per_row", [False, True])
@pytest.mark.parametrize("norm", [True, False])
@pytest.mark.parametrize("dim,inter,tokens", [(2048, 8192, 2), (1536, 8192, 3), (96, 2080, 4), (544, 2048, 2),
                                              (1056, 64, 4), (2048, 10752, 3), (1536, 8224, 4),
                                              (1536, 8192, 13), (1056, 128, 5), (2048, 160, 16), (2080, 192, 17),
                                              (1568, 2272, 32), (4128, 256, 9),
                                              (5888, 160, 9), (5920, 160, 9), (4608, 160, 20), (4640, 160, 20)])
def test_ffn_few_tokens_equals_op_sequence(gpu_ctx, dim, inter, tokens, norm, per_row):
    shapes = ((inter, dim), (inter, dim), (dim, inter))
    w1, w3, w2 = (q4.Q4Matrix.from_blocks(n, k, synth.q4_blocks(50 + i + n, n, k), gpu_ctx)
                  for i, (n, k) in enumerate(shapes))
    x = synth.activations(60 + tokens, tokens, dim)
    x[tokens - 1, :32] = 0.0
    nw = (1 + 0.1 * synth.normal_f32(61, dim)).astype(np.float32) if norm else None
    q4.set_act_quant(q4.ActQuant.PerRow if per_row else q4.ActQuant.PerBlock, gpu_ctx)
    try:
        got = x.copy()
        q4.ffn_residual(w1, w3, w2, nw, 1e-5, got, tokens)
        normed = x.copy()
        if norm:
            q4.rms_norm(x, nw, 1e-5, normed, gpu_ctx)
        g, u = (np.zeros((tokens, inter), dtype=np.float32) for _ in range(2))
        q4.gemm_q4(w1, normed, g, tokens)
        q4.gemm_q4(w3, normed, u, tokens)
        q4.silu_mul(g, u, gpu_ctx)
        ref = x.copy()
        q4.gemm_q4_add(w2, g, ref, tokens)
    finally:
        q4.set_act_quant(q4.ActQuant.PerBlock, gpu_ctx)
        for w in (w1, w3, w2):
            w.free()
    assert np.array_equal(got.view(np.uint32), ref.view(np.uint32))


@pytest.mark.parametrize("dim,inter,tokens", [(6144, 6144, 9), (6176, 6144, 20)])
def test_ffn_few_tokens_long_rows(gpu_ctx, dim, inter, tokens):
    """Blocks of enough rows that the gate/up launch takes their longer rows too."""
    test_ffn_few_tokens_equals_op_sequence(gpu_ctx, dim, inter, tokens, True, False)


@pytest.mark.parametrize("warm,captured", [("PerBlock", "PerRow"), ("PerRow", "PerBlock")])
@pytest.mark.parametrize("dim,inter,tokens", [(1536, 8192, 2), (96, 2080, 4), (96, 10752, 3),
                                              (544, 2048, 4), (1056, 2272, 9), (64, 8224, 385)])
def test_ffn_shape_that_ran_once_is_captured_in_either_mode(dim, inter, tokens, warm, captured):
    """A block run eagerly in one act-quant mode needs no workspace to grow in the other: its capture
    is accepted and its replays equal an eager call."""
    import torch

    ctx = q4.Context(0)
    stream = torch.cuda.Stream()
    ctx.set_stream(stream.cuda_stream)
    w1, w3, w2 = (q4.Q4Matrix.from_blocks(n, k, synth.q4_blocks(n + i, n, k), ctx)
                  for i, (n, k) in enumerate(((inter, dim), (inter, dim), (dim, inter))))
    x = torch.from_numpy(synth.activations(60 + tokens, tokens, dim)).cuda()
    hidden = x.clone()
    torch.cuda.synchronize()

    def block():
        q4.ffn_residual(w1, w3, w2, None, 1e-5, hidden, tokens)

    with torch.cuda.stream(stream):
        q4.set_act_quant(q4.ActQuant[warm], ctx)
        block()
        q4.set_act_quant(q4.ActQuant[captured], ctx)
        torch.cuda.synchronize()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            block()
        got = []
        for _ in range(3):
            hidden.copy_(x)
            graph.replay()
            got.append(hidden.clone())
        hidden.copy_(x)
        block()
        torch.cuda.synchronize()
        for g in got:
            assert torch.equal(g.view(torch.int32), hidden.view(torch.int32))
    del graph
    for w in (w1, w3, w2):
        w.free()
    ctx.close()
