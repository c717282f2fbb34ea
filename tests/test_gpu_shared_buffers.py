"""lgh_q4_norm_gemv_dev on buffers that share memory: an output that is hidden itself equals the same
call into a buffer of its own, bit for bit, on the one-token, the two-to-four-token and the
matrix-core routes and on rows past one K slice, each with enough rows for many workgroups; and 2 to
64 tokens' projections that add to one output equal one call after another."""

import pytest

from llmhost_amd import q4, synth
from llmhost_amd._ffi import LGH_ADD_F32, LGH_ADD_F64, LGH_ASSIGN

pytestmark = pytest.mark.gpu


def _bits(t):
    import torch

    return t.view(torch.int32)


@pytest.mark.parametrize("mode", [LGH_ASSIGN, LGH_ADD_F64])
@pytest.mark.parametrize("k,tokens", [(2048, 1), (2048, 2), (1536, 4), (2048, 3), (512, 9), (2080, 4), (512, 70)])
def test_norm_gemv_in_place(gpu_ctx, k, tokens, mode):
    import torch

    w, w2 = (q4.Q4Matrix.from_blocks(n, k, synth.q4_blocks(n + s, n, k), gpu_ctx) for n, s in ((k, 1), (96, 2)))
    x = torch.from_numpy(synth.activations(tokens, tokens, k)).cuda()
    nw = torch.from_numpy(1 + 0.1 * synth.normal_f32(7, k)).float().cuda()
    ref, ref2, got2 = x.clone(), torch.zeros(tokens, 96, device="cuda"), torch.zeros(tokens, 96, device="cuda")
    q4.norm_gemv([w, w2], nw, 1e-5, x, [ref, ref2], tokens, mode)
    for _ in range(3):
        hidden = x.clone()
        got2.zero_()
        q4.norm_gemv([w, w2], nw, 1e-5, hidden, [hidden, got2], tokens, mode)
        torch.cuda.synchronize()
        assert torch.equal(_bits(hidden), _bits(ref)) and torch.equal(_bits(got2), _bits(ref2))
    for m in (w, w2):
        m.free()


@pytest.mark.parametrize("norm", [False, True])
@pytest.mark.parametrize("k,tokens", [(1536, 2), (2048, 4), (4096, 3), (8224, 4), (1536, 5), (2048, 40), (4096, 64)])
def test_norm_gemv_adds_to_one_output(gpu_ctx, k, tokens, norm):
    import torch

    n = 1536
    ws = [q4.Q4Matrix.from_blocks(n, k, synth.q4_blocks(s, n, k), gpu_ctx) for s in (1, 2, 3)]
    x = torch.from_numpy(synth.activations(tokens, tokens, k)).cuda()
    nw = torch.from_numpy(1 + 0.1 * synth.normal_f32(7, k)).float().cuda() if norm else None
    ref = torch.from_numpy(synth.activations(9, tokens, n)).cuda()
    start = ref.clone()
    for w in ws:
        q4.norm_gemv([w], nw, 1e-5, x, [ref], tokens, LGH_ADD_F32)
    for _ in range(3):
        got = start.clone()
        q4.norm_gemv(ws, nw, 1e-5, x, [got, got, got], tokens, LGH_ADD_F32)
        torch.cuda.synchronize()
        assert torch.equal(_bits(got), _bits(ref))
    for w in ws:
        w.free()
