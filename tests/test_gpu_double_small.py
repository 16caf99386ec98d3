"""Double products of 16 x 16 tiles (csrc/gemm_f64.hip, d_small_tile): edges of the tile, contractions around one, two and more stages
of 64 k, operands that 16-byte chunks do not fit, batches, the gradients of an inner product and the heads in one launch."""
import numpy as np
import pytest

from oracle import attention_ref as R
from tests.test_gpu_double import devd  # noqa: F401

pytestmark = pytest.mark.gpu

BOUND = lambda k: 2.0 ** -53 * (4 + np.sqrt(k))  # noqa: E731  (of the sum of |a| |b|)


@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k", [(16, 16, 2), (14, 18, 62), (18, 14, 64), (32, 2, 66), (2, 150, 128), (50, 34, 130), (66, 48, 194), (256, 256, 1024), (17, 15, 63),
                                   (33, 31, 3), (1, 5, 1023), (31, 65, 129)])
def test_edges(devd, m, n, k, tA, tB):  # noqa: F811
    rng = np.random.default_rng(m + n + k)
    a, b, c = rng.standard_normal((m, k)), rng.standard_normal((k, n)), rng.standard_normal((m, n))
    ha, hb, hc = devd.put((a.T if tA else a).copy()), devd.put((b.T if tB else b).copy()), devd.put(c)
    scale = np.abs(a) @ np.abs(b)
    devd.cuda.gemm(tA, tB, m, n, k, -0.5, ha, hb, 1.0, hc)
    assert (np.abs(devd.get(hc, (m, n)) - (c - 0.5 * (a @ b))) <= BOUND(k) * (scale + np.abs(c))).all()
    devd.cuda.gemm(tA, tB, m, n, k, 1.0, ha, hb, 0.0, hc)
    assert (np.abs(devd.get(hc, (m, n)) - a @ b) <= BOUND(k) * scale).all()


@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False)])
@pytest.mark.parametrize("outer,m,n,k", [(8, 128, 64, 128), (3, 17, 66, 70), (5, 30, 33, 15)])
def test_batches(devd, outer, m, n, k, tA, tB):  # noqa: F811
    rng = np.random.default_rng(outer)
    a, b = rng.standard_normal((outer, m, k)), rng.standard_normal((outer, k, n))
    hc = devd.zeros(outer * m * n)
    devd.cuda.matmul(outer, m, n, k, devd.put((a.transpose(0, 2, 1) if tA else a).copy()), devd.put((b.transpose(0, 2, 1) if tB else b).copy()), hc, 1.0, tA, tB)
    assert (np.abs(devd.get(hc, (outer, m, n)) - a @ b) <= BOUND(k) * (np.abs(a) @ np.abs(b))).all()


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("m,n,k", [(12, 3, 3), (64, 64, 64), (256, 256, 256), (256, 1024, 256), (33, 131, 65), (1, 40, 36), (7, 500, 12)])
def test_gradients_of_an_inner_product(devd, m, n, k, bias):  # noqa: F811
    rng = np.random.default_rng(m + n + k)
    x, w, dy, dw, db, dx = (rng.standard_normal(s) for s in ((m, k), (n, k), (m, n), (n, k), (n,), (m, k)))
    for accumulate in (False, True):
        hdw, hdb, hdx = devd.put(dw), devd.put(db), devd.put(dx)
        devd.cuda.LinearBackward(m, n, k, devd.put(x), devd.put(w), devd.put(dy), hdw, hdb if bias else 0, hdx, accumulate)
        assert (np.abs(devd.get(hdw, (n, k)) - (dw + dy.T @ x)) <= BOUND(m) * (np.abs(dy).T @ np.abs(x) + np.abs(dw))).all()
        assert (np.abs(devd.get(hdx, (m, k)) - (accumulate * dx + dy @ w)) <= BOUND(n) * (np.abs(dy) @ np.abs(w) + np.abs(dx))).all()
        assert (np.abs(devd.get(hdb, (n,)) - (db + bias * dy.sum(0))) <= BOUND(m) * (np.abs(dy).sum(0) + np.abs(db))).all()


def test_results_over_operands(devd):  # noqa: F811
    # what the calls one after the other, or by way of scratch memory, allow
    rng = np.random.default_rng(1)
    B, T, H, hs = 2, 16, 2, 16
    m, C = B * T, H * hs
    x, w, dy, w3 = rng.standard_normal((m, C)), rng.standard_normal((C, C)), rng.standard_normal((m, C)), rng.standard_normal((3 * C, C))
    hx, hdw, hdb = devd.put(x), devd.zeros(C * C), devd.zeros(C)
    devd.cuda.LinearBackward(m, C, C, hx, devd.put(w), devd.put(dy), hdw, hdb, hx)
    for h, want in ((hx, dy @ w), (hdw, dy.T @ x), (hdb, dy.sum(0))):
        assert np.abs(devd.get(h, want.shape) - want).max() <= 1e-13 * np.abs(want).max()
    hx, hk, hv = devd.put(x), devd.zeros(m * C), devd.zeros(m * C)
    devd.cuda.QkvProjHeads(B, T, H, hs, hx, devd.put(w3), 0, hx, hk, hv)
    for h, want in zip((hx, hk, hv), (x @ w3.T).reshape(B, T, 3, H, hs).transpose(2, 0, 3, 1, 4)):
        assert np.abs(devd.get(h, want.shape) - want).max() <= 1e-13 * np.abs(want).max()
    hx = devd.put(x)
    devd.cuda.LinearForward(m, C, C, hx, devd.put(w), 0, hx, T, H)
    want = (x @ w.T).reshape(B, T, H, hs).transpose(0, 2, 1, 3)
    assert np.abs(devd.get(hx, want.shape) - want).max() <= 1e-13 * np.abs(want).max()


@pytest.mark.parametrize("B,T,H,hs,rope", [(1, 33, 2, 16, False), (2, 30, 3, 6, True), (2, 128, 4, 64, True), (3, 7, 1, 5, False)])
def test_into_heads(devd, B, T, H, hs, rope):  # noqa: F811
    C, rng = H * hs, np.random.default_rng(T)
    x, w, b = rng.standard_normal((B * T, C)), rng.standard_normal((3 * C, C)), rng.standard_normal(3 * C)
    hq = [devd.zeros(B * T * C) for _ in range(3)]
    hr = devd.cuda.CreateRope(0, 0, B * T * C, B, T, H, hs, 10000.0) if rope else 0
    hx, hw, hb = devd.put(x), devd.put(w), devd.put(b)
    devd.cuda.QkvProjHeads(B, T, H, hs, hx, hw, hb, *hq, hr)
    ref = x @ w.T + b
    for i, h in enumerate(hq):
        third = ref.reshape(B, T, 3, H, hs)[:, :, i]
        want = R.rope_forward(third, T, H, hs, dtype=np.float64).reshape(B, T, H, hs) if rope and i < 2 else third
        # the rotation's angles and factors are fp32: an angle below T is off by 2^-24 of itself twice (the frequency, the product), a pair
        # of values by that times its length, and the factors by 2^-24 each
        tol = np.sqrt(2) * (2 * T + 2) * 2.0 ** -24 if rope and i < 2 else 1e-13
        assert np.abs(devd.get(h, (B, H, T, hs)).transpose(0, 2, 1, 3) - want).max() <= tol * np.abs(ref).max()
    hy = devd.zeros(B * T * C)
    devd.cuda.LinearForward(B * T, C, C, hx, hw, hb, hy, T, H)
    want = ref[:, :C].reshape(B, T, H, hs).transpose(0, 2, 1, 3)
    assert np.abs(devd.get(hy, want.shape) - want).max() <= 1e-13 * np.abs(ref).max()
    if hr:
        devd.cuda.FreeRope(hr)
