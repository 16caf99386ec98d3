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


# sizes that 256 x 288 tiles divide, fill one round of the chip, and 128 x 128 tiles would not: the smallest contraction taken,
# one that ends an odd number of stages later, and the two ways the sizes can be met
@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("m,n,k", [(8192, 2304, 256), (14592, 1152, 288), (8192, 2304, 252)])
def test_one_round_of_wide_tiles(dev, m, n, k, bias):
    rng = np.random.default_rng(k)
    x, w, b = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (n, k), (n,)))
    hx, hw, hb, hy = dev.put(x), dev.put(w), dev.put(b), dev.zeros(m * n)
    ref = x.astype(np.float64) @ w.T.astype(np.float64)
    dev.cuda.gemm(False, True, m, n, k, -0.5, hx, hw, 0.0, hy)
    assert np.abs(dev.get(hy, (m, n)) + 0.5 * ref).max() / np.abs(ref).max() < 2e-6
    dev.cuda.LinearForward(m, n, k, hx, hw, hb if bias else 0, hy)
    assert np.abs(dev.get(hy, (m, n)) - ref - (b if bias else 0)).max() / np.abs(ref).max() < 2e-6


@pytest.mark.parametrize("rope", [False, True])
def test_one_round_of_wide_tiles_into_heads(dev, rope):
    from oracle import attention_ref as R
    B, T, H, hs = 16, 512, 12, 64
    C = H * hs
    rng = np.random.default_rng(5)
    x, w, b = (rng.standard_normal(s).astype(np.float32) for s in ((B * T, C), (3 * C, C), (3 * C,)))
    hq = [dev.zeros(B * T * C) for _ in range(3)]
    hr = dev.cuda.CreateRope(0, 0, B * T * C, B, T, H, hs, 10000.0) if rope else 0
    dev.cuda.QkvProjHeads(B, T, H, hs, dev.put(x), dev.put(w), dev.put(b), *hq, hr)
    ref = (x.astype(np.float64) @ w.T.astype(np.float64) + b).reshape(B, T, 3, H, hs)
    for i, h in enumerate(hq):
        want = R.rope_forward(ref[:, :, i], T, H, hs, dtype=np.float64).reshape(B, T, H, hs) if rope and i < 2 else ref[:, :, i]
        assert np.abs(dev.get(h, (B, H, T, hs)).transpose(0, 2, 1, 3) - want).max() <= (1e-4 if rope else 4e-6) * np.abs(ref).max()
    if hr:
        dev.cuda.FreeRope(hr)
