"""The 256 x 256 tiles of the batched GEMM (both operands through LDS) and the gate/up
pair they run in one launch."""
import ctypes

import numpy as np
import pytest
import torch

import blockpack as bp
from test_gpu_parity import assert_rows_close, tight_bound, to_dev

pytestmark = pytest.mark.gpu
Q4_0, Q5_0, Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K = 2, 6, 8, 10, 11, 12, 13, 14
TYPES = [Q4_0, Q5_0, Q8_0, Q2_K, Q3_K, Q4_K, Q5_K, Q6_K]


def _with_env(monkeypatch, env, t, raws, n, k, run):
    """run(lib, ctx, handles) in a context that read `env`."""
    from lightbulb_amd import _lib
    L = _lib.lib()
    for key, v in env.items():
        monkeypatch.setenv(key, v)
    ctx = ctypes.c_void_p()
    _lib.check(L.lbq_init(0, ctypes.byref(ctx)))
    for key in env:
        monkeypatch.delenv(key)
    hs = []
    try:
        for raw in raws:
            h = ctypes.c_void_p()
            _lib.check(L.lbq_weight_wrap_device(ctx, t, n, k, raw.data_ptr(), raw.numel(), ctypes.byref(h)))
            hs.append(h)
        return run(L, ctx, hs)
    finally:
        for h in hs:
            L.lbq_weight_destroy(h)
        L.lbq_ctx_destroy(ctx)


def _blocks(oracle, rng, t, n, k, dev):
    raw = bp.random_blocks(rng, t, n * k // oracle.block_size(t), d_scale=1e-3)
    return raw, to_dev(raw, dev)


@pytest.mark.parametrize("t", TYPES)
# one block and several; row and column tiles whole, one over, one short
@pytest.mark.parametrize("m,n,k", [(256, 256, 256), (257, 300, 768), (511, 33, 1280), (700, 512, 512)])
def test_square_tiles(oracle, lbq, dev, t, m, n, k, monkeypatch):
    rng = np.random.default_rng(31 * t + m)
    raw, rd = _blocks(oracle, rng, t, n, k, dev)
    x = rng.standard_normal((m, k)).astype(np.float32)
    xd, y = to_dev(x, dev), torch.full((m, n), float("nan"), device=dev)

    def run(L, ctx, hs):
        assert L.lbq_qmatmul_f32(ctx, hs[0], xd.data_ptr(), m, y.data_ptr(), None) == 0
        torch.cuda.synchronize()

    torch.cuda.synchronize()
    _with_env(monkeypatch, {"LBQ_GEMM_BIG": "square"}, t, [rd], n, k, run)
    rows = sorted({0, 31, 32, 127, 128, 255, m // 2, m - 1})
    assert_rows_close(y[rows].cpu().numpy(), oracle.qmatmul(t, raw, n, k, x[rows], nthreads=8).astype(np.float64),
                      tight_bound(t, m))


@pytest.mark.parametrize("t", [Q4_0, Q8_0, Q3_K, Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("m,n,k,off", [(300, 8300, 512, 0), (513, 5600, 256, 0), (257, 8256, 768, 1)])
def test_square_pair(oracle, lbq, dev, t, m, n, k, off, monkeypatch):
    # the plan's own choice (more than 128 tiles of 128 outputs): the bits of the two
    # products on the same tiles and the product launch; x 16-byte aligned and not
    rng = np.random.default_rng(17 * t + m)
    (rg, gd), (ru, ud) = _blocks(oracle, rng, t, n, k, dev), _blocks(oracle, rng, t, n, k, dev)
    base = to_dev(rng.standard_normal(m * k + off).astype(np.float32), dev)
    xd = base[off:].reshape(m, k)
    outs = []

    def run(L, ctx, hs):
        y = torch.full((m, n), float("nan"), device=dev)
        torch.cuda.synchronize()
        assert L.lbq_gate_up_silu_f32(ctx, hs[0], hs[1], xd.data_ptr(), m, y.data_ptr(), None) == 0
        torch.cuda.synchronize()
        outs.append(y.cpu().numpy())

    _with_env(monkeypatch, {}, t, [gd, ud], n, k, run)
    _with_env(monkeypatch, {"LBQ_GEMM_BIG": "square", "LBQ_GEMM_PAIR_OFF": "1"}, t, [gd, ud], n, k, run)
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    rows = [0, 128, 255, 256, m - 1]
    x = xd.cpu().numpy()[rows]
    g = oracle.qmatmul(t, rg, n, k, x, nthreads=8).astype(np.float64)
    u = oracle.qmatmul(t, ru, n, k, x, nthreads=8).astype(np.float64)
    # each factor within the fp16 operands' bound of its row; silu' is at most 1.1
    assert_rows_close(outs[0][rows], g / (1.0 + np.exp(-g)) * u, 2e-3)


def test_square_group_mixes_kernels(oracle, lbq, dev):
    # one pre-pass for weights of different n, one on the square tiles and one not
    from lightbulb_amd.quantized import GgmlDType, QMatMul, QTensor, qmatmul_group
    rng = np.random.default_rng(5)
    m, k = 384, 512
    ns = (17000, 300)
    for t in (Q4_K, Q6_K):
        raws = [_blocks(oracle, rng, t, n, k, dev) for n in ns]
        qs = [QMatMul.from_qtensor(QTensor(d, GgmlDType(t), (n, k))) for (_, d), n in zip(raws, ns)]
        xd = to_dev(rng.standard_normal((m, k)).astype(np.float32), dev)
        for y, q in zip(qmatmul_group(qs, xd), qs):
            assert torch.equal(y, q.forward(xd))
        rows = [0, 200, m - 1]
        ref = oracle.qmatmul(t, raws[0][0], ns[0], k, xd.cpu().numpy()[rows], nthreads=8).astype(np.float64)
        assert_rows_close(qs[0].forward(xd)[rows].cpu().numpy(), ref, tight_bound(t, m))


@pytest.mark.parametrize("t", [Q8_0, Q4_K, Q6_K])
@pytest.mark.parametrize("k", [512, 4352])
@pytest.mark.parametrize("off", [0, 1])
def test_norm_then_square_pair(oracle, lbq, dev, t, k, off, monkeypatch):
    # the norm inside the pre-pass (off = 1: the norm weight only 4-byte aligned, a launch of
    # its own) and the pair after it: the bits of the two products and the product launch
    rng = np.random.default_rng(19 * t + k)
    m, n = 300, 8300
    (rg, gd), (ru, ud) = _blocks(oracle, rng, t, n, k, dev), _blocks(oracle, rng, t, n, k, dev)
    x = (3.0 * rng.standard_normal((m, k))).astype(np.float32)
    w = (1.0 + 0.1 * rng.standard_normal(k)).astype(np.float32)
    xd, wd = to_dev(x, dev), to_dev(np.concatenate([np.zeros(off), w]).astype(np.float32), dev)[off:]
    outs = []

    def run(L, ctx, hs):
        y = torch.full((m, n), float("nan"), device=dev)
        torch.cuda.synchronize()
        assert L.lbq_rmsnorm_gate_up_silu_f32(ctx, hs[0], hs[1], xd.data_ptr(), wd.data_ptr(), 1e-5, m, y.data_ptr(), None) == 0
        torch.cuda.synchronize()
        outs.append(y.cpu().numpy())

    _with_env(monkeypatch, {}, t, [gd, ud], n, k, run)
    _with_env(monkeypatch, {"LBQ_GEMM_BIG": "square", "LBQ_GEMM_PAIR_OFF": "1"}, t, [gd, ud], n, k, run)
    assert np.array_equal(outs[0].view(np.uint32), outs[1].view(np.uint32))
    rows = [0, 128, 255, 256, m - 1]
    x64 = x[rows].astype(np.float64)
    xn = (x64 / np.sqrt((x64 ** 2).mean(1, keepdims=True) + 1e-5) * w).astype(np.float32)
    g = oracle.qmatmul(t, rg, n, k, xn, nthreads=8).astype(np.float64)
    u = oracle.qmatmul(t, ru, n, k, xn, nthreads=8).astype(np.float64)
    # the fp16 operands' bound of test_square_pair, and of x_norm rounded in f32 another
    # way: codes at a tie move by one, 2^-7 of a block's largest for few of its values
    assert_rows_close(outs[0][rows], g / (1.0 + np.exp(-g)) * u, 2e-3)
