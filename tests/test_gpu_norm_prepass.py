"""RMS norm in registers (rows of k % 4 == 0 up to 16384 values) and inside the batched
GEMM's operand pre-pass."""
import numpy as np
import pytest
import torch

import blockpack as bp
from test_gpu_parity import assert_rows_close, tight_bound, to_dev

pytestmark = pytest.mark.gpu
Q4_0, Q4_1, Q8_0, Q4_K, Q6_K = 2, 3, 8, 12, 14


@pytest.mark.parametrize("k", [4, 1000, 2048, 2052, 4096, 8192, 8196, 16384, 16388, 1003])
def test_rms_norm(lbq, dev, k):
    # each register count and its edges, and the rows it does not take
    from lightbulb_amd.quantized import rms_norm
    rng = np.random.default_rng(k)
    x = rng.standard_normal((5, k)).astype(np.float32)
    w = rng.standard_normal(k).astype(np.float32)
    y = rms_norm(to_dev(x, dev), to_dev(w, dev), 1e-5).cpu().numpy()
    x64 = x.astype(np.float64)
    ref = x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + 1e-5) * w
    # a sum of k squares in f32 (relative error below k/64 2^-24 by the partial sums), a
    # square root, a division and a product
    assert np.abs(y - ref).max() <= (k / 64 + 8) * 2.0 ** -24 * np.abs(ref).max()


@pytest.mark.parametrize("t", [Q4_0, Q4_1, Q8_0, Q4_K, Q6_K])
# 256 threads with one to four passes, 1024 threads (long rows), and rows it does not fuse
@pytest.mark.parametrize("m,k,off", [(130, 1024, 0), (130, 4352, 0), (130, 8448, 0), (1100, 12544, 0), (1100, 4096, 0),
                                     (140, 2048, 1), (100, 768, 0)])
def test_norm_in_prepass(oracle, lbq, dev, t, m, k, off):
    from lightbulb_amd.quantized import GgmlDType, QMatMul, QTensor, rms_norm, rmsnorm_gate_up_silu, rmsnorm_qmatmul_group
    rng = np.random.default_rng(3 * t + m + k)
    n = 96
    raws = [bp.random_blocks(rng, t, n * k // oracle.block_size(t), d_scale=1e-3) for _ in range(2)]
    qs = [QMatMul.from_qtensor(QTensor(to_dev(r, dev), GgmlDType(t), (n, k))) for r in raws]
    x = to_dev((3.0 * rng.standard_normal(m * k + off)).astype(np.float32), dev)[off:].reshape(m, k)
    w = to_dev((1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32), dev)
    ys = rmsnorm_qmatmul_group(qs, x, w, 1e-5)
    h = rmsnorm_gate_up_silu(qs[0], qs[1], x, w, 1e-5).cpu().numpy()
    rows = [0, m // 2, m - 1]
    xn = rms_norm(x, w, 1e-5).cpu().numpy()[rows]
    refs = [oracle.qmatmul(t, r, n, k, xn, nthreads=8).astype(np.float64) for r in raws]
    for y, ref in zip(ys, refs):
        assert_rows_close(y.cpu().numpy()[rows], ref, tight_bound(t, m))
    g, u = refs
    assert_rows_close(h[rows], g / (1.0 + np.exp(-g)) * u, 2e-3)


def _rms_in_order(x, eps):
    """sqrt(mean(x^2) + eps) of a row in f32, summed as row_rms does: 256 threads' chains of
    fused multiply-adds, quads, the quads of a row of 16 (0 + 3, then 2 + 1), rows, waves."""
    ss = np.zeros(256, np.float32)
    u = np.zeros(-(-len(x) // 256) * 256, np.float32)
    u[:len(x)] = x
    for v in u.reshape(-1, 256).astype(np.longdouble):
        ss = (v * v + ss).astype(np.float32)  # the product is exact, one rounding
    q = ss.reshape(-1, 4)
    q = ((q[:, 0] + q[:, 1]) + (q[:, 2] + q[:, 3])).reshape(-1, 4)
    r = ((q[:, 0] + q[:, 3]) + (q[:, 2] + q[:, 1])).reshape(-1, 4)
    w = ((r[:, 0] + r[:, 1]) + r[:, 2]) + r[:, 3]
    s = ((w[0] + w[1]) + w[2]) + w[3]
    return np.sqrt(s / np.float32(len(x)) + np.float32(eps), dtype=np.float32)


@pytest.mark.parametrize("k", [1, 255, 1000, 2048, 2052, 4096, 8192, 16384, 16388, 40000])
def test_rms_norm_sum_order(lbq, dev, k):
    # bit for bit, whichever kernel and alignment serves the row
    from lightbulb_amd.quantized import rms_norm
    rng = np.random.default_rng(k)
    x, w = rng.standard_normal((3, k)).astype(np.float32), rng.standard_normal(k).astype(np.float32)
    want = np.stack([r / _rms_in_order(r, 1e-5) * w for r in x])
    base = to_dev(np.concatenate([[0], x.reshape(-1)]).astype(np.float32), dev)
    for xd in (to_dev(x, dev), base[1:].reshape(3, k)):
        assert np.array_equal(rms_norm(xd, to_dev(w, dev), 1e-5).cpu().numpy(), want)


@pytest.mark.parametrize("t", [Q4_0, Q4_1, Q8_0, Q4_K, Q6_K])
# one to four passes of 256 threads, 1024 threads, the pair launch, separate norms
@pytest.mark.parametrize("m,n,k", [(130, 96, 1024), (130, 96, 4352), (130, 96, 8448), (130, 96, 12544), (66, 96, 4096),
                                   (1100, 96, 12544), (300, 8300, 4352), (20, 96, 768)])
def test_norm_in_prepass_is_norm_then_product(lbq, dev, t, m, n, k):
    # a norm inside another launch gives the bits of the norm by itself
    from lightbulb_amd.quantized import (GgmlDType, QMatMul, QTensor, gate_up_silu, qmatmul_group, rms_norm,
                                         rmsnorm_gate_up_silu, rmsnorm_qmatmul_group)
    rng = np.random.default_rng(5 * t + m + k)
    raws = [bp.random_blocks(rng, t, n * k // GgmlDType(t).block_size(), d_scale=1e-3) for _ in range(2)]
    qs = [QMatMul.from_qtensor(QTensor(to_dev(r, dev), GgmlDType(t), (n, k))) for r in raws]
    x = to_dev((3.0 * rng.standard_normal((m, k))).astype(np.float32), dev)
    w = to_dev((1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32), dev)
    xn = rms_norm(x, w, 1e-5)
    for a, b in zip(rmsnorm_qmatmul_group(qs, x, w, 1e-5), qmatmul_group(qs, xn)):
        assert torch.equal(a, b)
    assert torch.equal(rmsnorm_gate_up_silu(*qs, x, w, 1e-5), gate_up_silu(*qs, xn))
