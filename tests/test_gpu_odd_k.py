"""32-value block types whose k is no multiple of 256, at m > 8: integer block sums on the
fp16 matrix cores, against the oracle.

Bound: block sums and scale products are exact, so GPU and oracle differ by the f32
rounding of nb block terms each, 2^-24 of the running sum per term."""
import ctypes

import numpy as np
import pytest
import torch

import blockpack as bp
from test_gpu_parity import assert_rows_close, to_dev

pytestmark = pytest.mark.gpu
Q4_0, Q4_1, Q5_0, Q5_1, Q8_0 = 2, 3, 6, 7, 8
TYPES = [Q4_0, Q4_1, Q5_0, Q5_1, Q8_0]


def _qm(t, n, k, raw, dev):
    from lightbulb_amd.quantized import GgmlDType, QMatMul, QTensor
    return QMatMul.from_qtensor(QTensor(to_dev(raw, dev), GgmlDType(t), (n, k)))


@pytest.mark.parametrize("t", TYPES)
# row tiles of 32, 64 and 128 rows and their edges; column tiles of 256; one block, a
# stage (four blocks) less or more one, odd block counts, slices of k
@pytest.mark.parametrize("m,n,k", [(9, 1, 32), (32, 257, 96), (33, 31, 160), (64, 300, 288), (65, 513, 2080),
                                   (129, 64, 1184), (300, 40, 4128), (20, 1500, 992)])
def test_odd_k_shapes(oracle, lbq, dev, t, m, n, k):
    rng = np.random.default_rng(10 * t + m + n + k)
    raw = bp.random_blocks(rng, t, n * k // 32, d_scale=1e-2)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[rng.random(x.shape) < 0.01] *= 20
    y = _qm(t, n, k, raw, dev).forward(to_dev(x, dev)).cpu().numpy()
    ref = oracle.qmatmul(t, raw, n, k, x, nthreads=8).astype(np.float64)
    assert_rows_close(y, ref, max(k // 32, 4) * 2.0 ** -23)


@pytest.mark.parametrize("t", TYPES)
def test_odd_k_entry_points(oracle, lbq, dev, t):
    # x only 4-byte aligned, a pre-quantised handle, a group: the bits of forward()
    from lightbulb_amd.quantized import QActivation, qmatmul_group
    rng = np.random.default_rng(70 + t)
    m, k = 41, 1184
    raws = [bp.random_blocks(rng, t, n * k // 32, d_scale=1e-2) for n in (130, 37)]
    qa, qb = (_qm(t, n, k, r, dev) for n, r in zip((130, 37), raws))
    base = to_dev(rng.standard_normal(m * k + 4).astype(np.float32), dev)
    x = base[4:].reshape(m, k)
    ya, yb = qa.forward(x).cpu().numpy(), qb.forward(x).cpu().numpy()
    base[1:1 + m * k] = x.reshape(-1).clone()
    assert np.array_equal(qa.forward(base[1:1 + m * k].reshape(m, k)).cpu().numpy(), ya)
    x = x.clone()
    x.copy_(base[1:1 + m * k].reshape(m, k))
    assert np.array_equal(qa.forward_quantized(QActivation.for_weight(qa, m).quantize(x)).cpu().numpy(), ya)
    ga, gb = qmatmul_group([qa, qb], x)
    assert np.array_equal(ga.cpu().numpy(), ya) and np.array_equal(gb.cpu().numpy(), yb)


@pytest.mark.parametrize("t", TYPES)
def test_odd_k_nonfinite(lbq, dev, t):
    # infinities and NaN in x and in the scales: those of the decode kernel (m <= 8)
    rng = np.random.default_rng(90 + t)
    m, n, k = 24, 70, 352
    raw = bp.random_blocks(rng, t, n * k // 32, d_scale=1e-2).reshape(n, k // 32, -1).copy()
    raw[3, 2, :2] = np.array([np.inf], np.float16).view(np.uint8)
    raw[5, 10, :2] = np.array([np.nan], np.float16).view(np.uint8)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[1, 40], x[2, 351], x[4, 0], x[6] = np.inf, np.nan, 3e8, 0
    qm = _qm(t, n, k, raw.reshape(-1), dev)
    xd = to_dev(x, dev)
    y = qm.forward(xd).cpu().numpy()
    ref = np.concatenate([qm.forward(xd[i:i + 8]).cpu().numpy() for i in range(0, m, 8)])
    assert np.array_equal(np.isnan(y), np.isnan(ref)) and np.array_equal(np.isinf(y), np.isinf(ref))
    fin = np.isfinite(ref)
    assert np.array_equal(y[~fin & ~np.isnan(ref)], ref[~fin & ~np.isnan(ref)])
    assert np.linalg.norm(y[fin] - ref[fin]) <= 11 * 2.0 ** -23 * np.linalg.norm(ref[fin])


def test_odd_k_noalloc_limit_and_capture(oracle, lbq, dev):
    # the operands beyond the fixed scratch: row chunks; graph replays between eager calls
    from lightbulb_amd.quantized import context
    rng = np.random.default_rng(99)
    n, k, m = 2000, 2080, 4096
    raw = bp.random_blocks(rng, Q8_0, n * k // 32, d_scale=1e-2)
    qm = _qm(Q8_0, n, k, raw, dev)
    x = rng.standard_normal((m, k)).astype(np.float32)
    xd, y = to_dev(x, dev), torch.empty(m, n, device=dev)
    st = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
    rows = [0, 1000, m - 1]
    ref = oracle.qmatmul(Q8_0, raw, n, k, x[rows], nthreads=8).astype(np.float64)
    for mm in (m, 12000):
        if mm != m:
            xd = torch.cat([xd] * 3)[:mm].contiguous()
            y = torch.empty(mm, n, device=dev)
        assert lbq.lbq_qmatmul_f32_noalloc(context(dev), qm._handle, xd.data_ptr(), mm, y.data_ptr(), st) == 0
        assert_rows_close(y[rows].cpu().numpy(), ref, 65 * 2.0 ** -23)
    xs = xd[:50].contiguous()
    want = qm.forward(xs)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        yg = qm.forward(xs)
    for _ in range(3):
        yg.zero_()
        qm.forward(xd[50:90].contiguous())
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(yg, want)
