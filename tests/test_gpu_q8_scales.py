"""Q8_0 weights at m > 8 whose block scales lie far apart in a row: each value enters the
matrix cores as one f16 rounding of code times scale, also in the blocks with the
smallest (subnormal) scales, which the large ones must not push out of f16's range.

x is whole numbers with a 127 in every block, so its codes and operands are exact, and it
is zero where the weight's scale is large: only the small blocks show.  Bound: half an ulp
of f16 for each product and of f32 for each of the k/16 sums.
"""
import numpy as np
import pytest
import torch

from test_gpu_parity import to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [40, 100, 200, 333])  # k-sliced, wide and tall tiles
@pytest.mark.parametrize("small", [3 * 2.0 ** -24, 1.2998046875 * 2.0 ** -14, 0.0137])
def test_q8_0_small_scales_beside_large(lbq, dev, m, small):
    from lightbulb_amd.quantized import GgmlDType, QMatMul, QTensor
    rng = np.random.default_rng(5)
    n, k = 300, 1024
    d = np.full((n, k // 32), small, np.float16)
    big = rng.random((n, k // 32)) < 0.3
    big[:, 0], big[:, 5] = True, False
    big[1:] = big[0]
    d[big] = 1.37
    codes = rng.integers(-128, 128, (n, k // 32, 32)).astype(np.int8)
    raw = np.concatenate([d.view(np.uint8).reshape(n, -1, 2), codes.view(np.uint8)], axis=2).reshape(-1)
    qm = QMatMul.from_qtensor(QTensor(to_dev(raw, dev), GgmlDType(8), (n, k)))
    x = rng.integers(-126, 127, (m, k // 32, 32)).astype(np.float32)
    x[:, :, 7] = 127
    x[:, big[0]] = 0
    x = x.reshape(m, k)
    y = qm.forward(to_dev(x, dev)).cpu().numpy().astype(np.float64)
    w = (codes.astype(np.float64) * d.astype(np.float64)[:, :, None]).reshape(n, k)
    ref, mass = x.astype(np.float64) @ w.T, np.abs(x).astype(np.float64) @ np.abs(w).T
    assert (np.abs(y - ref) <= (2.0 ** -11 + k / 16 * 2.0 ** -24) * mass).all()
