"""Weights from f32 to blocks and back, and embedding rows, where their kernels branch."""
import numpy as np
import pytest
import torch

import blockpack as bp
from test_gpu_parity import gpu_quant_weights, to_dev

pytestmark = pytest.mark.gpu
F32, F16, BF16, Q4_0, Q8_0, Q4_K, Q5_K, Q6_K = 0, 1, 30, 2, 8, 12, 13, 14


def _hard_values(rng):
    """[rows, 256] that leave the code search's float side, or come close to it."""
    n = 64
    v = [rng.standard_normal((n, 256)), 20 * rng.standard_t(2, (n, 256)), np.zeros((n, 256)),
         np.full((n, 256), 0.7), np.full((n, 256), -0.7), -1.0 + 1e-7 * rng.integers(0, 3, (n, 256)),
         1.0 + 1e-7 * rng.integers(0, 9, (n, 256)), -1e3 - rng.random((n, 256)), rng.standard_normal((n, 256)) * 1e-38,
         rng.standard_normal((n, 256)) * 1e-44, rng.standard_normal((n, 256)) * 1e37,
         rng.standard_normal((n, 256)) * 10.0 ** rng.integers(-30, 30, (n, 1)),
         np.where(rng.random((n, 256)) < 0.05, rng.standard_normal((n, 256)), 0.0),
         np.round(rng.standard_normal((n, 256)) * 8) / 8]
    return np.concatenate(v).astype(np.float32)


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
def test_quantizer_hard_values_bit_exact(oracle, lbq, dev, t):
    rng = np.random.default_rng(t)
    w = _hard_values(rng)
    with np.errstate(all="ignore"):
        ref = oracle.quantize_weights(t, w)
    assert np.array_equal(gpu_quant_weights(t, w, dev), ref)
    # in an order that mixes kinds within a wave
    w = w[rng.permutation(len(w))]
    with np.errstate(all="ignore"):
        ref = oracle.quantize_weights(t, w)
    assert np.array_equal(gpu_quant_weights(t, w, dev), ref)


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
def test_quantizer_alignment_and_tail(oracle, lbq, dev, t):
    # values 4-byte aligned only; a last workgroup of one block
    from lightbulb_amd.quantized import quantize_tensor
    rng = np.random.default_rng(20 + t)
    w = rng.standard_normal((33, 256)).astype(np.float32)
    base = to_dev(np.concatenate([[0], w.reshape(-1)]).astype(np.float32), dev)
    assert np.array_equal(quantize_tensor(base[1:], t).cpu().numpy(), oracle.quantize_weights(t, w))


@pytest.mark.parametrize("t", [F32, F16, BF16, Q4_0, Q8_0, Q4_K, Q6_K])
@pytest.mark.parametrize("blocks", [1, 3, 4, 64, 65, 1023])
def test_dequantize_tails(oracle, lbq, dev, t, blocks):
    # partial waves (64 runs of 16 values) and partial groups of four dense values
    from lightbulb_amd.quantized import GgmlDType, dequantize_tensor
    rng = np.random.default_rng(blocks)
    if t in (F32, F16, BF16):
        n = 16 * blocks - 3
        f = rng.standard_normal(n).astype(np.float32)
        v = torch.from_numpy(f).to({F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}[t])
        got = dequantize_tensor(v.view(torch.uint8).to(dev), GgmlDType(t), n).cpu()
        assert torch.equal(got, v.to(torch.float32))
        return
    raw = bp.random_blocks(rng, t, blocks, d_scale=1e-2)
    n = blocks * oracle.block_size(t)
    got = dequantize_tensor(to_dev(raw, dev), GgmlDType(t), n).cpu().numpy()
    assert np.array_equal(got.view(np.uint32), oracle.dequantize(t, raw).reshape(-1).view(np.uint32))


@pytest.mark.parametrize("t", [F32, F16, BF16, Q4_0, Q4_K])
@pytest.mark.parametrize("k,count", [(256, 1), (256, 5), (1280, 7), (4096, 3)])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32])
def test_embedding_rows(lbq, dev, t, k, count, dtype):
    from lightbulb_amd.quantized import GgmlDType, QEmbedding, QTensor
    rng = np.random.default_rng(k + count)
    n = 40
    if t in (F32, F16, BF16):
        raw = torch.from_numpy(rng.standard_normal(n * k).astype(np.float32)).to(
            {F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}[t]).view(torch.uint8).numpy()
    else:
        raw = bp.random_blocks(rng, t, n * k // GgmlDType(t).block_size(), d_scale=1e-2)
    qt = QTensor(to_dev(raw, dev), GgmlDType(t), (n, k))
    table = qt.dequantize().cpu().numpy()
    ids = rng.integers(0, n, count)
    ids[count // 2] = n if count > 1 else ids[0]
    got = QEmbedding(qt).forward(torch.from_numpy(ids).to(dtype)).cpu().numpy()
    for i, r in enumerate(ids):
        assert np.isnan(got[i]).all() if r == n else np.array_equal(got[i], table[r])
    if dtype == torch.int64:  # ids no int32 holds are outside the table too
        far = torch.tensor([2 ** 32, -1, 2 ** 40 + 1], device=dev)
        assert torch.isnan(QEmbedding(qt).forward(far)).all()
