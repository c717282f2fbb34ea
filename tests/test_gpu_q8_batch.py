"""The Q8_0 head over several tokens (one weight pass per 64 tokens) against the oracle's q8_apply
(crates/llm-engine/src/weights.rs:194-227), at the edges of its tiles: rows that end inside a
16-row tile and off a float4, odd block counts, rows one block past an LDS stage, every number of
token tiles, several passes.  Tolerance: the output tolerance of every route (summation order)."""

import numpy as np
import pytest

from llmhost_amd import q4, synth

from .conftest import assert_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,tokens", [(8197, 1056, 13), (8192, 2048, 16), (8200, 2080, 17), (8194, 4128, 33),
                                        (16384, 512, 64), (8193, 1024, 100), (32768, 1536, 3)])
@pytest.mark.parametrize("norm", [False, True])
def test_q8_batch_matches_oracle(gpu_ctx, oracle, n, k, tokens, norm):
    blocks = synth.q8_blocks(n + k, n, k)
    x = synth.activations(tokens, tokens, k)
    x[tokens // 2] = 0.0
    w = q4.Q8Matrix.from_blocks(n, k, blocks, gpu_ctx)
    y = np.zeros((tokens, n), dtype=np.float32)
    if norm:
        nw = (1 + 0.1 * synth.normal_f32(7, k)).astype(np.float32)
        q4.q8_norm_apply(w, nw, 1e-5, x, tokens, y)
        x = np.stack([oracle.rms_norm(r, nw, 1e-5) for r in x])
    else:
        q4.q8_apply(w, x, tokens, y)
    ref = oracle.q8_apply(blocks, n, k, x, tokens, threads=8).reshape(tokens, n)
    w.free()
    assert_close(y, ref, what=f"q8 {n}x{k} m={tokens}")


def test_q8_batch_keeps_tokens_apart(gpu_ctx):
    """An infinite activation reaches its own token only, whatever stage and tile it sits in."""
    n, k, tokens = 8192, 2080, 20
    w = q4.Q8Matrix.from_blocks(n, k, synth.q8_blocks(3, n, k), gpu_ctx)
    x = synth.activations(4, tokens, k)
    y, z = (np.zeros((tokens, n), dtype=np.float32) for _ in range(2))
    q4.q8_apply(w, x, tokens, y)
    x[3, k - 1] = np.inf
    q4.q8_apply(w, x, tokens, z)
    w.free()
    keep = np.arange(tokens) != 3
    assert np.array_equal(y[keep], z[keep])
    assert not np.isfinite(z[3]).any()


def test_q8_batch_under_capture_without_a_workspace(oracle):
    """A captured call whose image workspace would have to grow takes the GEMV instead."""
    import torch

    n, k, tokens = 8192, 2048, 16
    blocks = synth.q8_blocks(5, n, k)
    ctx = q4.Context(0)
    stream = torch.cuda.Stream()
    ctx.set_stream(stream.cuda_stream)
    w = q4.Q8Matrix.from_blocks(n, k, blocks, ctx)
    xh = synth.activations(6, tokens, k)
    x = torch.from_numpy(xh).cuda()
    y = torch.zeros(tokens, n, device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        q4.q8_apply(w, x, tokens, y)
    ref = oracle.q8_apply(blocks, n, k, xh, tokens, threads=8).reshape(tokens, n)
    for _ in range(3):
        y.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert_close(y.cpu().numpy(), ref, what="captured q8")
    del graph
    w.free()
    ctx.close()


def test_q8_batch_graph_survives_growth_and_trim(oracle):
    """A captured pass keeps its workspace when a later call grows it and when it is trimmed."""
    import torch

    n, k, tokens = 8192, 2048, 16
    blocks = synth.q8_blocks(5, n, k)
    ctx = q4.Context(0)
    stream = torch.cuda.Stream()
    ctx.set_stream(stream.cuda_stream)
    w = q4.Q8Matrix.from_blocks(n, k, blocks, ctx)
    w4 = q4.Q4Matrix.from_blocks(64, 8192, synth.q4_blocks(6, 64, 8192), ctx)
    xh = synth.activations(6, tokens, k)
    x = torch.from_numpy(xh).cuda()
    y = torch.zeros(tokens, n, device="cuda")
    x4, y4 = torch.randn(600, 8192, device="cuda"), torch.zeros(600, 64, device="cuda")
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.stream(stream):
        q4.q8_apply(w, x, tokens, y)  # sizes the workspace
        torch.cuda.synchronize()
        with torch.cuda.graph(graph, stream=stream):
            q4.q8_apply(w, x, tokens, y)
    ref = oracle.q8_apply(blocks, n, k, xh, tokens, threads=8).reshape(tokens, n)
    for step in range(3):
        with torch.cuda.stream(stream):
            if step == 1:
                q4.gemm_q4(w4, x4, y4, 600)
            if step == 2:
                ctx.trim()
            junk = torch.full((1 << 22,), float("nan"), device="cuda")  # what was freed is written over
            y.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
        assert_close(y.cpu().numpy(), ref, what=f"replay {step}")
        del junk
    del graph
    w.free()
    w4.free()
    ctx.close()
