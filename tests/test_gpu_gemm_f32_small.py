"""fp32 products of 32 x 32 tiles (csrc/gemm_f32.hip, gemm_f32_small_kernel): edges of the tile, contractions around one, two and more
stages of 64 k, batches, both ends of the causal ranges, the epilogues."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BOUND = lambda k: 2.0 ** -24 * (4 + np.sqrt(k))  # noqa: E731  (of the sum of |a| |b|: one rounding per two k, the parts' and the result's)

SHAPES = [(32, 32, 4), (28, 36, 124), (36, 28, 128), (64, 4, 132), (4, 300, 256), (100, 68, 260), (132, 96, 384), (32, 3072, 388), (200, 1000, 300),
          (288, 292, 1024), (1024, 288, 288)]


@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_edges(dev, m, n, k, tA, tB):
    rng = np.random.default_rng(m + n + k)
    a, b, c = (rng.standard_normal(s, dtype=np.float32) for s in ((m, k), (k, n), (m, n)))
    ha, hb, hc = dev.put((a.T if tA else a).copy()), dev.put((b.T if tB else b).copy()), dev.put(c)
    want, scale = a.astype(np.float64) @ b.astype(np.float64), np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64))
    dev.cuda.gemm(tA, tB, m, n, k, -0.5, ha, hb, 1.0, hc)
    assert (np.abs(dev.get(hc, (m, n)) - (c - 0.5 * want)) <= BOUND(k) * (0.5 * scale + np.abs(c))).all()
    dev.cuda.gemm(tA, tB, m, n, k, 1.0, ha, hb, 0.0, hc)
    assert (np.abs(dev.get(hc, (m, n)) - want) <= BOUND(k) * scale).all()


@pytest.mark.parametrize("tA,tB", [(False, True), (True, False)])
@pytest.mark.parametrize("outer,m,n,k", [(24, 256, 48, 256), (3, 36, 132, 140), (7, 64, 64, 16)])
def test_batches(dev, outer, m, n, k, tA, tB):
    rng = np.random.default_rng(outer)
    a, b = rng.standard_normal((outer, m, k), dtype=np.float32), rng.standard_normal((outer, k, n), dtype=np.float32)
    ha, hb = dev.put((a.transpose(0, 2, 1) if tA else a).copy()), dev.put((b.transpose(0, 2, 1) if tB else b).copy())
    hc = dev.zeros(outer * m * n)
    dev.cuda.matmul(outer, m, n, k, ha, hb, hc, 1.0, tA, tB)
    a, b = a.astype(np.float64), b.astype(np.float64)
    assert (np.abs(dev.get(hc, (outer, m, n)) - a @ b) <= BOUND(k) * (np.abs(a) @ np.abs(b))).all()


@pytest.mark.parametrize("outer,T,hs", [(24, 256, 48), (3, 1023, 63), (30, 96, 40), (2, 33, 31)])
def test_causal_operands(dev, outer, T, hs):
    from mycaffe_amd.cudadnn import load_library
    from tests.test_gpu_gemm_f32_split import causal_products
    assert load_library().MCH_GemmFloatRoute(T, hs, T, outer, 1) % 4 == load_library().MCH_GemmFloatRoute(hs, T, T, outer, 1) % 4 == 2
    causal_products(dev, outer, T, hs)


@pytest.mark.parametrize("B,T,H,hs,rope", [(1, 33, 2, 16, False), (2, 30, 6, 48, True), (4, 256, 6, 48, True)])
def test_into_heads(dev, B, T, H, hs, rope):
    from oracle import attention_ref as R
    C, rng = H * hs, np.random.default_rng(T)
    x, w, b = (rng.standard_normal(s, dtype=np.float32) for s in ((B * T, C), (3 * C, C), (3 * C,)))
    hq = [dev.zeros(B * T * C) for _ in range(3)]
    hr = dev.cuda.CreateRope(0, 0, B * T * C, B, T, H, hs, 10000.0) if rope else 0
    hx, hw, hb = dev.put(x), dev.put(w), dev.put(b)
    dev.cuda.QkvProjHeads(B, T, H, hs, hx, hw, hb, *hq, hr)
    ref = x.astype(np.float64) @ w.T.astype(np.float64) + b
    for i, h in enumerate(hq):
        third = ref.reshape(B, T, 3, H, hs)[:, :, i]
        want = R.rope_forward(third, T, H, hs, dtype=np.float64).reshape(B, T, H, hs) if rope and i < 2 else third
        # the rotation's angles are fp32
        assert np.abs(dev.get(h, (B, H, T, hs)).transpose(0, 2, 1, 3) - want).max() <= (1e-4 if rope else 4e-6) * np.abs(ref).max()
    hy = dev.zeros(B * T * 3 * C)
    dev.cuda.LinearForward(B * T, 3 * C, C, hx, hw, hb, hy)
    assert np.abs(dev.get(hy, ref.shape) - ref).max() <= 4e-6 * np.abs(ref).max()
    if hr:
        dev.cuda.FreeRope(hr)


def test_infinities_and_nan(dev):
    rng = np.random.default_rng(2)
    m, n, k = 96, 64, 260
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    a[5, 259], a[40, 0], a[95, 130] = np.inf, np.nan, -np.inf
    hc = dev.zeros(m * n)
    dev.cuda.gemm(False, False, m, n, k, 1.0, dev.put(a), dev.put(b), 0.0, hc)
    got = dev.get(hc, (m, n))
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[[5, 95]], want[[5, 95]].astype(np.float32))
    rest = np.setdiff1d(np.arange(m), [5, 40, 95])
    assert np.isfinite(got[rest]).all()


# odd sizes and operands that begin anywhere: 4 bytes a lane
@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k", [(33, 31, 3), (12, 3, 12), (65, 130, 127), (129, 34, 129), (31, 97, 257), (1, 5, 1023)])
def test_odd_sizes(dev, m, n, k, tA, tB):
    rng = np.random.default_rng(m + n + k)
    a, b, c = (rng.standard_normal(s, dtype=np.float32) for s in ((m, k), (k, n), (m, n)))
    ha, hb, hc = dev.put((a.T if tA else a).copy()), dev.put((b.T if tB else b).copy()), dev.put(c)
    want, scale = a.astype(np.float64) @ b.astype(np.float64), np.abs(a.astype(np.float64)) @ np.abs(b.astype(np.float64))
    dev.cuda.gemm(tA, tB, m, n, k, 2.0, ha, hb, 1.0, hc)
    assert (np.abs(dev.get(hc, (m, n)) - (c + 2 * want)) <= BOUND(k) * (2 * scale + np.abs(c))).all()


# the gradients of an inner product as one launch: the longer contraction in either, edges of tiles and stages, with and without bias,
# data gradients that are added up; and memory that the three results or the operands share, which takes the calls one by one
@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("m,n,k", [(12, 3, 3), (12, 12, 3), (64, 64, 64), (1024, 288, 288), (256, 768, 96), (33, 131, 65), (1, 40, 36), (1030, 100, 32), (7, 500, 12)])
def test_gradients_of_an_inner_product(dev, m, n, k, bias):
    rng = np.random.default_rng(m + n + k)
    x, w, dy, dw, db, dx = (rng.standard_normal(s, dtype=np.float32) for s in ((m, k), (n, k), (m, n), (n, k), (n,), (m, k)))
    x64, w64, dy64 = (v.astype(np.float64) for v in (x, w, dy))
    for accumulate in (False, True):
        hdw, hdb, hdx = dev.put(dw), dev.put(db), dev.put(dx)
        dev.cuda.LinearBackward(m, n, k, dev.put(x), dev.put(w), dev.put(dy), hdw, hdb if bias else 0, hdx, accumulate)
        scale = np.abs(dy64).T @ np.abs(x64) + np.abs(dw)
        assert (np.abs(dev.get(hdw, (n, k)) - (dw + dy64.T @ x64)) <= BOUND(m) * scale).all()
        scale = np.abs(dy64) @ np.abs(w64) + np.abs(dx)
        assert (np.abs(dev.get(hdx, (m, k)) - (accumulate * dx + dy64 @ w64)) <= BOUND(n) * scale).all()
        want = db + dy64.sum(0) if bias else db
        assert (np.abs(dev.get(hdb, (n,)) - want) <= BOUND(m) * (np.abs(dy64).sum(0) + np.abs(db))).all()


def test_gradients_of_an_inner_product_in_shared_memory(dev):
    # the data gradient over the input, which the calls one after the other allow: the weight gradient has been made by then
    rng = np.random.default_rng(1)
    m = n = k = 64
    x, w, dy = (rng.standard_normal((64, 64), dtype=np.float32) for _ in range(3))
    hx, hdw, hdb = dev.put(x), dev.zeros(n * k), dev.zeros(n)
    dev.cuda.LinearBackward(m, n, k, hx, dev.put(w), dev.put(dy), hdw, hdb, hx)
    x, w, dy = (v.astype(np.float64) for v in (x, w, dy))
    for h, want in ((hx, dy @ w), (hdw, dy.T @ x), (hdb, dy.sum(0))):
        assert np.abs(dev.get(h, want.shape) - want).max() <= 1e-5 * np.abs(want).max()
