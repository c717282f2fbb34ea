"""Host-slice calls equal the same calls on device tensors bit for bit, on both sides of the pinned
staging's 512 KB per direction: inputs of exactly that size and one row more, the old output
counted in when the call adds, results too large, row counts that are no multiple of 4."""

import numpy as np
import pytest

from llmhost_amd import q4, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("add", [False, True])
@pytest.mark.parametrize("m,n,k", [(1, 1, 32), (1, 1537, 1536), (3, 70, 64), (64, 33, 2048), (65, 33, 2048),
                                   (16, 8192, 64), (17, 8192, 64), (40, 2049, 96)])
def test_host_call_equals_device_call(gpu_ctx, m, n, k, add):
    import torch

    w = q4.Q4Matrix.from_blocks(n, k, synth.q4_blocks(n + k, n, k), gpu_ctx)
    call = q4.gemm_q4_add if add else q4.gemm_q4
    for i in range(3):  # the staging buffer is used again, for other values
        x = synth.activations(m + 10 * i, m, k)
        hy = synth.activations(m + 10 * i + 1, m, n)
        dx, dz = torch.from_numpy(x).cuda(), torch.from_numpy(hy).cuda()
        call(w, x, hy, m)
        call(w, dx, dz, m)
        torch.cuda.synchronize()
        assert np.array_equal(hy.view(np.uint32), dz.cpu().numpy().view(np.uint32))
    w.free()


@pytest.mark.parametrize("n", [5, 8192, 65536, 70001])
def test_host_pair_and_q8_equal_device_calls(gpu_ctx, n):
    import torch

    k = 96
    x = synth.activations(9, 1, k)
    dx = torch.from_numpy(x).cuda()
    wg, wu = (q4.Q4Matrix.from_blocks(n, k, synth.q4_blocks(s, n, k), gpu_ctx) for s in (1, 2))
    w8 = q4.Q8Matrix.from_blocks(n, k, synth.q8_blocks(3, n, k), gpu_ctx)
    host = [np.zeros(n, dtype=np.float32) for _ in range(3)]
    dev = [torch.zeros(n, device="cuda") for _ in range(3)]
    q4.gemv_q4_pair(wg, wu, x, host[0], host[1])
    q4.q8_apply(w8, x, 1, host[2])
    q4.gemv_q4_pair(wg, wu, dx, dev[0], dev[1])
    q4.q8_apply(w8, dx, 1, dev[2])
    torch.cuda.synchronize()
    for h, d in zip(host, dev):
        assert np.array_equal(h.view(np.uint32), d.cpu().numpy().view(np.uint32))
    for w in (wg, wu, w8):
        w.free()


def test_host_calls_from_two_threads(gpu_ctx):
    """Two contexts on two threads: a call that finds the staging buffer taken uses pageable copies."""
    import threading

    n, k, calls = 1536, 1536, 40
    blocks = synth.q4_blocks(7, n, k)
    ref = np.zeros(n, dtype=np.float32)
    w0 = q4.Q4Matrix.from_blocks(n, k, blocks, gpu_ctx)
    x = synth.activations(8, 1, k)
    q4.gemv_q4(w0, x, ref)
    w0.free()
    bad = []

    def work():
        ctx = q4.Context(0)
        w = q4.Q4Matrix.from_blocks(n, k, blocks, ctx)
        for _ in range(calls):
            y = np.zeros(n, dtype=np.float32)
            q4.gemv_q4(w, x, y)
            if not np.array_equal(y, ref):
                bad.append(1)
        w.free()
        ctx.close()

    threads = [threading.Thread(target=work) for _ in range(2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
