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


def test_q8_batch_random_shapes(gpu_ctx, oracle):
    """Seeded sizes on both sides of the pass's rule, as the fuzz of the other routes."""
    rng = np.random.default_rng(20261204)
    for i in range(12):
        n, k, tokens = int(rng.integers(8192, 9300)), 32 * int(rng.integers(1, 140)), int(rng.integers(2, 131))
        print(f"[q8 fuzz {i}] n={n} k={k} tokens={tokens}", flush=True)
        blocks = synth.q8_blocks(i, n, k)
        x = synth.activations(100 + i, tokens, k)
        w = q4.Q8Matrix.from_blocks(n, k, blocks, gpu_ctx)
        y = np.zeros((tokens, n), dtype=np.float32)
        q4.q8_apply(w, x, tokens, y)
        w.free()
        ref = oracle.q8_apply(blocks, n, k, x, tokens, threads=8).reshape(tokens, n)
        assert_close(y, ref, what=f"q8 {n}x{k} m={tokens}")


@pytest.mark.parametrize("k,tokens", [(2080, 20), (2592, 48), (4128, 33), (8192, 16), (8192, 64), (16384, 40)])
def test_q8_batch_is_as_exact_as_one_token(gpu_ctx, oracle, k, tokens):
    """Rows of several tokens are no further from the 64-bit sums of the same codes than those of one
    token.  Over the 160000 outputs and more of a case an rms error varies by 0.2%, and the summation
    orders' errors lie within 4% of each other (one order whose chains grow with the row: 15% above
    at 256 blocks, 33% at 512)."""
    import torch

    n = 8192
    blocks = synth.q8_blocks(k, n, k)
    w = q4.Q8Matrix.from_blocks(n, k, blocks, gpu_ctx)
    x = synth.activations(tokens, tokens, k)
    dx = torch.from_numpy(x).cuda()
    many, one = (torch.zeros(tokens, n, device="cuda") for _ in range(2))
    q4.q8_apply(w, dx, tokens, many)
    for t in range(tokens):
        q4.q8_apply(w, dx[t], 1, one[t])
    qs, sa, _ = oracle.act_quantize(x, False)
    ex = torch.zeros(tokens, n, dtype=torch.float64, device="cuda")
    xq = torch.from_numpy(qs.reshape(tokens, -1, 32) * sa.astype(np.float64).reshape(tokens, -1, 1)).cuda()
    for r in range(0, n, 1024):
        b = blocks.reshape(n, -1)[r:r + 1024]
        wq = b["qs"].astype(np.float64) * b["scale"].view(np.float16).astype(np.float64)[..., None]
        ex[:, r:r + 1024] = xq.reshape(tokens, k) @ torch.from_numpy(wq).cuda().reshape(-1, k).T.contiguous()
    torch.cuda.synchronize()
    w.free()
    err = [((y.double() - ex).norm() / ex.norm()).item() for y in (many, one)]
    print(f"k={k} tokens={tokens}: {err[0]:.4e} against {err[1]:.4e}")
    assert err[0] <= 1.05 * err[1]


@pytest.mark.parametrize("n,k", [(8192, 512), (8192, 1024), (9216, 1536), (8448, 2048), (8456, 1024), (12288, 512)])
def test_q8_batch_rule(gpu_ctx, oracle, n, k):
    """On both sides of the rule that chooses between the pass and a GEMV row per token."""
    blocks = synth.q8_blocks(n + k, n, k)
    w = q4.Q8Matrix.from_blocks(n, k, blocks, gpu_ctx)
    x = synth.activations(5, 24, k)
    ref = oracle.q8_apply(blocks, n, k, x, 24, threads=8).reshape(24, n)
    for tokens in (2, 6, 7, 8, 9, 12, 13, 17, 20, 24):
        y = np.zeros((tokens, n), dtype=np.float32)
        q4.q8_apply(w, x[:tokens].copy(), tokens, y)
        assert_close(y, ref[:tokens], what=f"q8 {n}x{k} m={tokens}")
    w.free()


def test_q8_rows_past_one_launch_take_the_token_route(gpu_ctx):
    """K ranges of 32768 elements: several tokens equal one at a time, bit for bit."""
    n, k, tokens = 8192, 32800, 2
    w = q4.Q8Matrix.from_blocks(n, k, synth.q8_blocks(2, n, k), gpu_ctx)
    x = synth.activations(3, tokens, k)
    many, one = (np.zeros((tokens, n), dtype=np.float32) for _ in range(2))
    q4.q8_apply(w, x, tokens, many)
    for t in range(tokens):
        q4.q8_apply(w, x[t], 1, one[t])
    w.free()
    assert np.array_equal(many.view(np.uint32), one.view(np.uint32))


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
    """A call captured without an eager one before it runs the same pass as an eager one, bit for bit."""
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
    got = y.clone()
    q4.q8_apply(w, x, tokens, y)
    torch.cuda.synchronize()
    assert torch.equal(y.view(torch.int32), got.view(torch.int32))
    del graph
    w.free()
    ctx.close()


def test_q8_batch_graph_survives_growth_and_trim(oracle):
    """A captured pass keeps its image when later calls grow the context's workspaces and when they are trimmed."""
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


def _captured(stream, call):
    import torch

    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        call()
    return graph


def test_q4_graph_survives_a_larger_q8_call():
    """An eager Q8_0 pass whose image is larger than the workspace of a captured Q4 call leaves that
    workspace alone: what it would have freed is written over before the replay."""
    import torch

    ctx = q4.Context(0)
    stream = torch.cuda.Stream()
    ctx.set_stream(stream.cuda_stream)
    w4 = q4.Q4Matrix.from_blocks(96, 2048, synth.q4_blocks(6, 96, 2048), ctx)
    w8 = q4.Q8Matrix.from_blocks(8192, 2048, synth.q8_blocks(5, 8192, 2048), ctx)
    x4, x8 = (torch.from_numpy(synth.activations(m, m, 2048)).cuda() for m in (8, 64))
    y4, y8 = torch.zeros(8, 96, device="cuda"), torch.zeros(64, 8192, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        q4.gemm_q4(w4, x4, y4, 8)
        torch.cuda.synchronize()
        ref = y4.clone()
        graph = _captured(stream, lambda: q4.gemm_q4(w4, x4, y4, 8))
        for tokens in (32, 64, 33):
            q4.q8_apply(w8, x8[:tokens].contiguous(), tokens, y8[:tokens])
            junk = torch.full((1 << 22,), float("nan"), device="cuda")
            y4.zero_()
            torch.cuda.synchronize()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(y4.view(torch.int32), ref.view(torch.int32))
            del junk
    del graph
    w4.free()
    w8.free()
    ctx.close()


def test_q8_graphs_need_the_matrix_only():
    """Graphs of Q8_0 passes replayed on streams of their own, beside each other and eager calls of
    their context, and after the context is closed."""
    import torch

    n, k = 8200, 2080
    ctx = q4.Context(0)
    stream = torch.cuda.Stream()
    ctx.set_stream(stream.cuda_stream)
    w = q4.Q8Matrix.from_blocks(n, k, synth.q8_blocks(5, n, k), ctx)
    sizes = (16, 33, 64)
    xs = [torch.from_numpy(synth.activations(m, m, k)).cuda() for m in sizes]
    ys = [torch.zeros(m, n, device="cuda") for m in sizes]
    refs = [torch.zeros(m, n, device="cuda") for m in sizes]
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for x, r, m in zip(xs, refs, sizes):
            q4.q8_apply(w, x, m, r)
        torch.cuda.synchronize()
        graphs = [_captured(stream, lambda: q4.q8_apply(w, x, m, y)) for x, y, m in zip(xs[:2], ys, sizes)]
    side = [torch.cuda.Stream() for _ in graphs]
    for closed in (False, True):
        for _ in range(4):
            for y in ys:
                y.zero_()
            torch.cuda.synchronize()
            for _ in range(5):
                for g, s in zip(graphs, side):
                    with torch.cuda.stream(s):
                        g.replay()
                if not closed:
                    with torch.cuda.stream(stream):
                        q4.q8_apply(w, xs[2], 64, ys[2])
            torch.cuda.synchronize()
            for y, r in list(zip(ys, refs))[:2 if closed else 3]:
                assert torch.equal(y.view(torch.int32), r.view(torch.int32))
        if not closed:
            ctx.close()
    del graphs
    w.free()


def test_q8_capture_and_trim_give_the_workspace_back():
    """A captured pass holds its image, not the context's workspaces: trimming returns those, however
    often a pass is captured."""
    import torch

    n, k = 8192, 2048
    ctx = q4.Context(0)
    stream = torch.cuda.Stream()
    ctx.set_stream(stream.cuda_stream)
    w = q4.Q8Matrix.from_blocks(n, k, synth.q8_blocks(5, n, k), ctx)
    w4 = q4.Q4Matrix.from_blocks(64, 4096, synth.q4_blocks(6, 64, 4096), ctx)
    w4.prepare_gemm()
    m = 16384  # an activation image of over 100 MB
    x, y = torch.zeros(16, k, device="cuda"), torch.zeros(16, n, device="cuda")
    x4, y4 = torch.zeros(m, 4096, device="cuda"), torch.zeros(m, 64, device="cuda")
    torch.cuda.synchronize()
    graphs, free = [], []
    with torch.cuda.stream(stream):
        for _ in range(8):
            q4.gemm_q4(w4, x4, y4, m)
            q4.q8_apply(w, x, 16, y)
            torch.cuda.synchronize()
            graphs.append(_captured(stream, lambda: q4.q8_apply(w, x, 16, y)))
            ctx.trim()
            free.append(torch.cuda.mem_get_info()[0])
    assert free[0] - free[-1] < 100 << 20
    del graphs
    w.free()
    w4.free()
    ctx.close()


def test_q8_captured_images_are_bounded():
    """Past the bytes a matrix holds for captured calls a call takes the GEMV: rows as of one token."""
    import torch

    n, k, tokens, calls = 8192, 16384, 64, 60  # 1.1 MiB an image: 56 or 57 fit in 64 MiB
    ctx = q4.Context(0)
    stream = torch.cuda.Stream()
    ctx.set_stream(stream.cuda_stream)
    w = q4.Q8Matrix.from_blocks(n, k, synth.q8_blocks(5, n, k), ctx)
    x = torch.from_numpy(synth.activations(3, tokens, k)).cuda()
    ys = torch.zeros(calls, tokens, n, device="cuda")
    many, one = torch.zeros(tokens, n, device="cuda"), torch.zeros(tokens, n, device="cuda")
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        def step():
            for y in ys:
                q4.q8_apply(w, x, tokens, y)

        graph = _captured(stream, step)
        q4.q8_apply(w, x, tokens, many)
        for t in range(tokens):
            q4.q8_apply(w, x[t], 1, one[t])
        for _ in range(2):
            ys.zero_()
            graph.replay()
            torch.cuda.synchronize()
            for i in (0, 1, 40, 55):
                assert torch.equal(ys[i].view(torch.int32), many.view(torch.int32))
            for i in (58, 59):
                assert torch.equal(ys[i].view(torch.int32), one.view(torch.int32))
    del graph
    w.free()
    ctx.close()
