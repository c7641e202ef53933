"""Dense F16 / BF16 / F32 weights at m > 8: x (and an F32 weight) as 16-bit operands that
add up to it, on the matrix cores, against a float64 product.

Bound: every product is exact in the f32 accumulator (of an F32 weight's, what is left
out is below 2^-23 of it), so a row's relative L2 error is
that of adding P k/16 partial sums one after the other, each rounded to half an ulp
(2^-24) of the running sum: 2^-24 sqrt(P k / 16) for errors of independent sign, taken
twice, and never below f32's own rounding of a handful of steps.
"""
import ctypes

import numpy as np
import pytest
import torch

from test_gpu_parity import to_dev

pytestmark = pytest.mark.gpu
F32, F16, BF16 = 0, 1, 30


def _weight(t, n, k, rng, dev, w=None):
    from lightbulb_amd.quantized import GgmlDType, QMatMul, QTensor
    w = torch.from_numpy((rng.standard_normal((n, k)) * 0.05).astype(np.float32) if w is None else w)
    w = w.to({F32: torch.float32, F16: torch.float16, BF16: torch.bfloat16}[t])
    qm = QMatMul.from_qtensor(QTensor(w.reshape(-1).view(torch.uint8).to(dev), GgmlDType(t), (n, k)))
    return qm, w.to(torch.float64).numpy()


def _bound(t, k):
    return 2.0 ** -23 * max(4.0, ({F32: 6, F16: 2, BF16: 3}[t] * k / 16) ** 0.5)


def _assert_rows(y, ref, bound):
    err = np.linalg.norm(y.astype(np.float64) - ref, axis=1) / np.linalg.norm(ref, axis=1)
    assert err.max() <= bound, (err.max(), bound)


@pytest.mark.parametrize("t", [F16, BF16, F32])
# each row tile's edges (32, 64, 128 rows), column tiles of 128 and 256, k that is no
# multiple of a stage (64) or of two, one stage, slices of k and none
@pytest.mark.parametrize("m,n,k", [(9, 1, 8), (32, 130, 520), (33, 300, 4096), (64, 127, 72), (65, 257, 1000),
                                   (128, 640, 2048), (129, 4096, 64), (700, 8200, 200), (300, 64, 14336)])
def test_dense_mm_shapes(lbq, dev, t, m, n, k):
    rng = np.random.default_rng(m + n + k)
    qm, w = _weight(t, n, k, rng, dev)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[rng.random(x.shape) < 0.01] *= 20
    _assert_rows(qm.forward(to_dev(x, dev)).cpu().numpy(), x.astype(np.float64) @ w.T, _bound(t, k))


@pytest.mark.parametrize("t", [F16, BF16, F32])
def test_dense_mm_range_and_alignment(lbq, dev, t):
    # rows of very different size, subnormal rows, zero rows; x only 4-byte aligned
    rng = np.random.default_rng(7)
    m, n, k = 40, 200, 264
    qm, w = _weight(t, n, k, rng, dev)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x *= (10.0 ** rng.integers(-30, 30, (m, 1))).astype(np.float32)
    x[3] = 0
    base = to_dev(np.concatenate([[0], x.reshape(-1)]).astype(np.float32), dev)
    y = qm.forward(base[1:].reshape(m, k)).cpu().numpy()
    rows = [r for r in range(m) if r != 3]
    _assert_rows(y[rows], (x.astype(np.float64) @ w.T)[rows], _bound(t, k))
    assert not y[3].any()


@pytest.mark.parametrize("t", [F16, BF16, F32])
@pytest.mark.parametrize("m,n,k", [(20, 140, 64), (20, 140, 2048)])  # unsplit, and slices of k
def test_dense_mm_nonfinite(lbq, dev, t, m, n, k):
    # an infinity gives the infinities and NaN of the f32 product, nowhere else
    rng = np.random.default_rng(11)
    w = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[1, 5], x[2, 9], x[4, 60], x[4, 61] = np.inf, np.nan, np.inf, -np.inf
    x[6, 3] = 3e38
    w[7, 20], w[9, 5], w[11, 30] = np.inf, 0.0, np.nan
    x[8, 20] = 0.0
    qm, w = _weight(t, n, k, rng, dev, w)
    y = qm.forward(to_dev(x, dev)).cpu().numpy()
    with np.errstate(invalid="ignore", over="ignore"):
        ref = (x[:, None, :].astype(np.float64) * w[None]).sum(2)
        ref = np.where(np.abs(ref) > 3.4028235e38, np.copysign(np.inf, ref), ref)
    fin = np.isfinite(ref)
    assert np.array_equal(np.isnan(ref), np.isnan(y))
    assert np.array_equal(ref[~fin & ~np.isnan(ref)], y[~fin & ~np.isnan(ref)])
    for r in range(m):
        c = fin[r]
        if c.any():
            assert np.linalg.norm(y[r][c] - ref[r][c]) <= _bound(t, k) * np.linalg.norm(ref[r][c])


@pytest.mark.parametrize("t", [F16, F32])
def test_dense_mm_nonfinite_large_tiles(lbq, dev, t):
    # 128 x 256 tiles, the last row tile short: a lane's sixteen results are tested together
    rng = np.random.default_rng(19)
    m, n, k = 1430, 4096, 72
    w = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[1, 5], x[700, 9], x[1429, 60] = np.inf, np.nan, -np.inf
    w[7, 20], w[9, 5], w[4095, 30] = np.inf, 0.0, np.nan
    qm, w = _weight(t, n, k, rng, dev, w)
    y = qm.forward(to_dev(x, dev)).cpu().numpy()
    ref = (torch.from_numpy(x).double() @ torch.from_numpy(w).double().T).numpy()
    fin = np.isfinite(ref)
    assert np.array_equal(np.isnan(ref), np.isnan(y))
    assert np.array_equal(ref[~fin & ~np.isnan(ref)], y[~fin & ~np.isnan(ref)])
    _assert_rows(np.where(fin, y, 0)[fin.any(1)], np.where(fin, ref, 0)[fin.any(1)], _bound(t, k))


@pytest.mark.parametrize("t", [F16, F32])
def test_dense_mm_streams_growth_and_capture(lbq, dev, t):
    # the operand buffer: two streams in turn, a larger call while a captured graph
    # uses the smaller buffer, and replays between eager calls
    rng = np.random.default_rng(13)
    qm, w = _weight(t, 512, 1024, rng, dev)
    big, wb = _weight(t, 1024, 8192, rng, dev)
    x = rng.standard_normal((48, 1024)).astype(np.float32)
    xb = rng.standard_normal((600, 8192)).astype(np.float32)
    xd, xbd = to_dev(x, dev), to_dev(xb, dev)
    want, wantb = qm.forward(xd).cpu().numpy(), big.forward(xbd).cpu().numpy()
    _assert_rows(want, x.astype(np.float64) @ w.T, _bound(t, 1024))
    _assert_rows(wantb, xb.astype(np.float64) @ wb.T, _bound(t, 8192))
    s1, s2 = torch.cuda.Stream(), torch.cuda.Stream()
    ys = []
    torch.cuda.synchronize()
    for i in range(6):
        with torch.cuda.stream((s1, s2)[i % 2]):
            ys.append((big.forward(xbd), wantb) if i % 3 == 0 else (qm.forward(xd), want))
    torch.cuda.synchronize()
    for y, ref in ys:
        assert np.array_equal(y.cpu().numpy(), ref)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        yg = qm.forward(xd)
    huge, wh = _weight(t, 256, 16384, rng, dev)
    xh = to_dev(rng.standard_normal((2000, 16384)).astype(np.float32), dev)
    for _ in range(3):
        huge.forward(xh)
        yg.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert np.array_equal(yg.cpu().numpy(), want)


@pytest.mark.parametrize("t", [F16, F32])
def test_dense_mm_noalloc_beyond_scratch(lbq, dev, t):
    # operands beyond the fixed scratch: the f32 matrix cores, as accurate
    from lightbulb_amd.quantized import context
    rng = np.random.default_rng(17)
    n, k, m = 64, 16384, 1100
    qm, w = _weight(t, n, k, rng, dev)
    x = rng.standard_normal((m, k)).astype(np.float32)
    xd, y = to_dev(x, dev), torch.empty(m, n, device=dev)
    st = ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)
    assert lbq.lbq_qmatmul_f32_noalloc(context(dev), qm._handle, xd.data_ptr(), m, y.data_ptr(), st) == 0
    # k/2 sums of two products, one after the other
    _assert_rows(y.cpu().numpy(), x.astype(np.float64) @ w.T, 2.0 ** -23 * (k / 2) ** 0.5)


def _assert_outputs(y, x, w, k):
    """Each output by itself, against the sum of its own products' sizes: eight sums an MFMA
    of 16 k-values at most, errors of independent sign, taken twice (as _bound)."""
    x, w = x.astype(np.float64), w.astype(np.float64)
    err, size = np.abs(y - x @ w.T), np.abs(x) @ np.abs(w).T
    bound = 2.0 ** -23 * max(4.0, (8 * k / 16) ** 0.5)
    assert (err <= bound * size).all(), (err / size).max() / bound


@pytest.mark.parametrize("t", [F16, BF16, F32])
@pytest.mark.parametrize("m,n,k", [(9, 130, 256), (64, 127, 2048), (300, 300, 512), (700, 8200, 200)])
@pytest.mark.parametrize("big", [1e6, 1e9, 1e20, 1e30])
def test_dense_mm_range_within_rows(lbq, dev, t, m, n, k, big):
    # one large value a row whose weights are zero: the row's other products are the result
    rng = np.random.default_rng(m + n + k)
    w = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    w[:, [3, k // 2]] = 0
    qm, w = _weight(t, n, k, rng, dev, w)
    x = rng.standard_normal((m, k)).astype(np.float32)
    x[:, 3] = big * np.where(np.arange(m) % 2, 1, -1)
    x[::3, 3], x[::3, k // 2] = 0, big
    y = qm.forward(to_dev(x, dev)).cpu().numpy()
    x[:, [3, k // 2]] = 0
    _assert_outputs(y, x, w, k)


def test_dense_mm_f32_products(lbq, dev):
    # one product an output: within a rounding or two of the f32 product (half an ulp, 2^-24,
    # for the first pieces' sum and again for its sum with the others; what is left out is
    # 2^-32), values whose pieces are as large as they get
    rng = np.random.default_rng(23)
    m, n, k = 300, 300, 72
    bits = lambda s: (0x3f800000 | 0xff7f | (rng.integers(0, 128, s) << 16)).astype(np.uint32).view(np.float32)
    x, w = np.zeros((m, k), np.float32), np.zeros((n, k), np.float32)
    x[:, 5], w[:, 5] = bits(m), bits(n)
    w[:, 6] = rng.standard_normal(n)  # meets zeros
    qm, wd = _weight(F32, n, k, rng, dev, w)
    ref = x.astype(np.float64) @ wd.T
    y = qm.forward(to_dev(x, dev)).cpu().numpy()
    assert np.abs(y / ref - 1).max() <= 2.1 * 2.0 ** -24


_SIZES = [(1e-36, 1.0), (1e-36, 1e4), (1e-42, 1e4), (1e-36, 1e20), (1e20, 1e-36), (1e30, 1e-42), (1e30, 1.0), (1e36, 1e-3)]


@pytest.mark.parametrize("m,n,k", [(9, 130, 256), (64, 127, 2048), (300, 300, 512), (700, 8200, 200)])
@pytest.mark.parametrize("t,xs,ws", [(t, xs, ws) for t in (F16, BF16, F32) for xs, ws in _SIZES
                                     if t == F32 or ws in (1.0, 1e4) or (t == BF16 and ws >= 1e-3)])
def test_dense_mm_small_and_large_values(lbq, dev, t, m, n, k, xs, ws):
    # down to f32's last bit and up to its largest, on either side
    rng = np.random.default_rng(m + k)
    qm, w = _weight(t, n, k, rng, dev, (rng.standard_normal((n, k)) * ws).astype(np.float32))
    x = (rng.standard_normal((m, k)) * xs).astype(np.float32)
    y = qm.forward(to_dev(x, dev)).cpu().numpy()
    x, w = x.astype(np.float64), w.astype(np.float64)
    size = np.abs(x) @ np.abs(w).T
    # a result below the normal range has f32's fixed spacing there, 2^-149
    bound = np.maximum(2.0 ** -23 * max(4.0, (8 * k / 16) ** 0.5) * size, 2.0 ** -149)
    assert (np.abs(y - x @ w.T) <= bound).all()


@pytest.mark.parametrize("t", [F16, BF16, F32])
# one product a tile and slices of k; tiles of 32, 64, 128 rows and 128 x 256, short ones
@pytest.mark.parametrize("m,n,k", [(20, 140, 64), (50, 70, 136), (40, 300, 2048), (300, 300, 1000), (1430, 4096, 72)])
def test_dense_mm_nonfinite_batch(lbq, dev, t, m, n, k):
    # x and W with NaN and infinities throughout; the finite outputs beside them keep their bits
    rng = np.random.default_rng(29)
    w = (rng.standard_normal((n, k)) * 0.05).astype(np.float32)
    x = rng.standard_normal((m, k)).astype(np.float32)
    qm, wf = _weight(t, n, k, rng, dev, w)
    clean = qm.forward(to_dev(x, dev)).cpu().numpy()
    x2, w2 = x.copy(), w.copy()
    x2[1::3, 7], x2[2::3, k - 1] = np.nan, np.inf
    w2[3::5, 2], w2[:, k - 1] = -np.inf, np.where(np.arange(n) % 2, 0, w2[:, k - 1])
    qm2, wd = _weight(t, n, k, rng, dev, w2)
    with np.errstate(invalid="ignore"):
        ref = (torch.from_numpy(x2).double() @ torch.from_numpy(wd).T).numpy()
    y = qm2.forward(to_dev(x2, dev)).cpu().numpy()
    fin = np.isfinite(ref)
    assert np.array_equal(np.isnan(ref), np.isnan(y))
    assert np.array_equal(ref[~fin & ~np.isnan(ref)], y[~fin & ~np.isnan(ref)])
    same = fin & (np.arange(n) % 2 == 0)  # rows of W that did not change
    assert np.array_equal(y[same], clean[same])
    x2[:] = np.nan
    assert np.isnan(qm2.forward(to_dev(x2, dev)).cpu().numpy()).all()


@pytest.mark.parametrize("t", [F16, F32])
def test_dense_mm_streams_side_by_side(lbq, dev, t):
    # many streams, a graph captured on one of them and replayed on another, none ordered
    # against the others: every call's own result
    rng = np.random.default_rng(31)
    qm, w = _weight(t, 640, 2048, rng, dev)
    xs = [rng.standard_normal((m, 2048)).astype(np.float32) for m in (40, 60, 130, 300)]
    xd = [to_dev(x, dev) for x in xs]
    want = [qm.forward(x).cpu().numpy() for x in xd]
    for x, y in zip(xs, want):
        _assert_rows(y, x.astype(np.float64) @ w.T, _bound(t, 2048))
    streams = [torch.cuda.Stream() for _ in range(20)]
    graphs = []
    for i in (0, 2):  # two graphs from one stream, the second larger
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=streams[0]):
            graphs.append((g, qm.forward(xd[i]), want[i]))
    torch.cuda.synchronize()
    for _ in range(4):
        ys = []
        for g, yg, _ in graphs:
            yg.zero_()
        torch.cuda.synchronize()
        for j, st in enumerate(streams):
            with torch.cuda.stream(st):
                if j in (1, 3):
                    graphs[j // 2][0].replay()
                ys += [(qm.forward(xd[i]), i) for i in ((j + 1) % 4, (j + 3) % 4)]
        torch.cuda.synchronize()
        for g, yg, ref in graphs:
            assert np.array_equal(yg.cpu().numpy(), ref)
        for y, i in ys:
            assert np.array_equal(y.cpu().numpy(), want[i])


def test_dense_mm_beside_a_capture(lbq, dev):
    # a call that has to allocate, in another thread and on another stream than a capture in
    # progress (whose mode forbids allocations elsewhere by default), does not end the capture
    import threading

    rng = np.random.default_rng(37)
    qm, w = _weight(F16, 256, 1024, rng, dev)
    x = rng.standard_normal((64, 1024)).astype(np.float32)
    xd, y, ys = to_dev(x, dev), torch.empty(64, 256, device=dev), torch.empty(64, 256, device=dev)
    want = qm.forward(xd).cpu().numpy()
    other = torch.cuda.Stream()
    ctx, h, rc = ctypes.c_void_p(), ctypes.c_void_p(), []
    assert lbq.lbq_init(0, ctypes.byref(ctx)) == 0
    data = qm.qtensor().data
    assert lbq.lbq_weight_wrap_device(ctx, F16, 256, 1024, data.data_ptr(), data.numel(), ctypes.byref(h)) == 0
    try:
        def beside():
            rc.append(lbq.lbq_qmatmul_f32(ctx, h, xd.data_ptr(), 64, ys.data_ptr(), ctypes.c_void_p(other.cuda_stream)))

        torch.cuda.synchronize()
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g):
            th = threading.Thread(target=beside)
            th.start()
            th.join()
            assert lbq.lbq_qmatmul_f32(ctx, h, xd.data_ptr(), 64, y.data_ptr(),
                                       ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream)) == 0
        for _ in range(3):
            y.zero_()
            g.replay()
            torch.cuda.synchronize()
            assert np.array_equal(y.cpu().numpy(), want)
        assert rc == [0] and np.array_equal(ys.cpu().numpy(), want)
    finally:
        torch.cuda.synchronize()
        lbq.lbq_weight_destroy(h)
        lbq.lbq_ctx_destroy(ctx)


@pytest.mark.parametrize("t", [F16, BF16, F32])
# one stage of k and one value more; k without slices on 64-row tiles, their edges, and with slices
@pytest.mark.parametrize("m,n,k", [(100, 520, 64), (4100, 1030, 64), (100, 520, 72), (129, 130, 504), (1000, 500, 256),
                                   (129, 130, 512), (4000, 1100, 128)])
def test_dense_mm_short_k(lbq, dev, t, m, n, k):
    rng = np.random.default_rng(m + k)
    qm, w = _weight(t, n, k, rng, dev)
    x = rng.standard_normal((m, k)).astype(np.float32)
    y = qm.forward(to_dev(x, dev)).cpu().numpy()
    rows = sorted({0, 31, 32, 63, 64, 127, 128, m // 2, m - 1} & set(range(m)))
    _assert_rows(y[rows], x[rows].astype(np.float64) @ w.T, _bound(t, k))


def test_dense_mm_per_thread_streams(lbq, dev):
    # hipStreamPerThread: one handle, a stream of its own in each thread
    import threading

    from lightbulb_amd.quantized import context
    rng = np.random.default_rng(41)
    n, k = 1024, 2048
    qm, w = _weight(F16, n, k, rng, dev)
    xs = [rng.standard_normal((m, k)).astype(np.float32) for m in (300, 200, 100, 40)]
    xd = [to_dev(x, dev) for x in xs]
    ys = [torch.empty(x.shape[0], n, device=dev) for x in xs]
    torch.cuda.synchronize()
    rc = []

    def calls(i):
        for _ in range(5):
            rc.append(lbq.lbq_qmatmul_f32(context(dev), qm._handle, xd[i].data_ptr(), xs[i].shape[0], ys[i].data_ptr(),
                                          ctypes.c_void_p(2)))

    threads = [threading.Thread(target=calls, args=(i,)) for i in range(4)]
    for th in threads:
        th.start()
    for th in threads:
        th.join()
    torch.cuda.synchronize()
    assert rc == [0] * 20
    for x, y in zip(xs, ys):  # k/2 sums of two products, one after the other
        _assert_rows(y.cpu().numpy(), x.astype(np.float64) @ w.T, 2.0 ** -23 * (k / 2) ** 0.5)
