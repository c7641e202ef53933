"""Captured calls whose context's buffers are outgrown afterwards: a replay still finds its own."""
import ctypes

import numpy as np
import pytest
import torch

import blockpack as bp
from test_gpu_parity import to_dev

pytestmark = pytest.mark.gpu
Q5_0, Q8_0, Q4_K, Q6_K = 6, 8, 12, 14


def _raw(oracle, rng, t, n, k, dev):
    return to_dev(bp.random_blocks(rng, t, n * k // oracle.block_size(t), d_scale=1e-3), dev)


# (small call, large call): odd widths (operands and partials), the pre-pass and split
# partials, pre-quantised codes (x 4-byte aligned), the matrix-core decode
@pytest.mark.parametrize("t,m,n,k,off,big", [(Q8_0, 50, 300, 1184, 0, (3000, 600, 4096)), (Q5_0, 50, 300, 4128, 1, (3000, 600, 4128)),
                                             (Q4_K, 100, 512, 4096, 0, (3000, 600, 4096)), (Q6_K, 50, 512, 2048, 1, (3000, 600, 2048)),
                                             (Q4_K, 16, 1024, 4096, 0, (3000, 600, 4096))])
def test_replay_after_growth(oracle, lbq, dev, t, m, n, k, off, big):
    rng = np.random.default_rng(t + m)
    ctx, hs = ctypes.c_void_p(), []
    assert lbq.lbq_init(0, ctypes.byref(ctx)) == 0

    def weight(n, k):
        raw, h = _raw(oracle, rng, t, n, k, dev), ctypes.c_void_p()
        assert lbq.lbq_weight_wrap_device(ctx, t, n, k, raw.data_ptr(), raw.numel(), ctypes.byref(h)) == 0
        hs.append((h, raw))
        return h

    def call(h, x, y):
        st = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
        assert lbq.lbq_qmatmul_f32(ctx, h, x.data_ptr(), x.shape[0], y.data_ptr(), st) == 0

    try:
        w, wb = weight(n, k), weight(big[1], big[2])
        x = to_dev(rng.standard_normal(m * k + off).astype(np.float32), dev)[off:].reshape(m, k)
        y, yg = torch.empty(m, n, device=dev), torch.empty(m, n, device=dev)
        call(w, x, y)
        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            call(w, x, yg)
        for i in range(3):
            # every buffer of the small call outgrown; what takes freed memory is watched
            xb = torch.randn(big[0] * 4 ** i // 4 + off, big[2], device=dev).reshape(-1)[off:]
            xb = xb[:xb.numel() // big[2] * big[2]].reshape(-1, big[2])
            yb = torch.empty(xb.shape[0], big[1], device=dev)
            call(wb, xb, yb)
            kept = [torch.full((1 << 18,), 7.0, device=dev) for _ in range(64)]
            before = yb.clone()
            yg.zero_()
            torch.cuda.synchronize()
            g.replay()
            torch.cuda.synchronize()
            assert torch.equal(yg, y) and torch.equal(yb, before)
            assert all(bool((b == 7.0).all()) for b in kept)
            yb.zero_()
            call(wb, xb, yb)
            torch.cuda.synchronize()
            assert torch.equal(yb, before)
    finally:
        torch.cuda.synchronize()
        for h, _ in hs:
            lbq.lbq_weight_destroy(h)
        lbq.lbq_ctx_destroy(ctx)
