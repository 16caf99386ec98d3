"""The fp32 GEMM kernel (csrc/gemm_f32.hip) where it can go wrong: edges of its tiles, contractions that end inside a stage or
inside a 16-byte chunk, operands whose rows are not aligned, contractions cut into parts, batches, beta."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

SHAPES = [(64, 64, 32), (65, 67, 33), (1, 129, 100), (129, 1, 65), (127, 191, 31), (128, 192, 96), (130, 198, 70), (200, 72, 288), (33, 1001, 48),
          (72, 132, 2500), (96, 96, 5001), (2048, 260, 36), (260, 2052, 68), (3, 9, 5)]


@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_gemm_edges(dev, m, n, k, tA, tB):
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    a, b, c = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (k, n), (m, n)))
    ha, hb = dev.put((a.T if tA else a).copy()), dev.put((b.T if tB else b).copy())
    want = a.astype(np.float64) @ b.astype(np.float64)
    for alpha, beta in ((1.0, 0.0), (0.5, 1.0)):
        hc = dev.put(c)
        dev.cuda.gemm(tA, tB, m, n, k, alpha, ha, hb, beta, hc)
        ref = alpha * want + beta * c
        err = np.abs(dev.get(hc, (m, n)) - ref).max() / np.abs(ref).max()
        assert err < 2e-6 * max(1.0, np.sqrt(k) / 16), err


@pytest.mark.parametrize("outer,m,n,k", [(3, 65, 48, 130), (5, 32, 96, 20), (2, 130, 3, 64), (24, 40, 40, 33)])
@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False)])
def test_batched_matmul_edges(dev, outer, m, n, k, tA, tB):
    rng = np.random.default_rng(outer + m)
    a, b = rng.standard_normal((outer, m, k)).astype(np.float32), rng.standard_normal((outer, k, n)).astype(np.float32)
    ha = dev.put((a.transpose(0, 2, 1) if tA else a).copy())
    hb = dev.put((b.transpose(0, 2, 1) if tB else b).copy())
    hc = dev.zeros(outer * m * n)
    dev.cuda.matmul(outer, m, n, k, ha, hb, hc, 1.0, tA, tB)
    ref = a.astype(np.float64) @ b.astype(np.float64)
    assert np.abs(dev.get(hc, (outer, m, n)) - ref).max() / np.abs(ref).max() < 2e-6


@pytest.mark.parametrize("m,n,k", [(70, 66, 36), (5, 50, 700), (64, 64, 4096), (300, 7, 33)])
def test_linear_forward_edges(dev, m, n, k):
    rng = np.random.default_rng(n)
    x, w, b = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (n, k), (n,)))
    hy = dev.zeros(m * n)
    dev.cuda.LinearForward(m, n, k, dev.put(x), dev.put(w), dev.put(b), hy)
    ref = x.astype(np.float64) @ w.T.astype(np.float64) + b
    assert np.abs(dev.get(hy, (m, n)) - ref).max() / np.abs(ref).max() < 4e-6
