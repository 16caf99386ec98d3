"""The calls that stand for several of a block's (ids 2005 - 2011), in every storage type, against float64 formulas: rows in
registers and rows too long for them, head sizes for each vector width, row counts on both sides of the split of a sum."""
import numpy as np
import pytest

from mycaffe_amd.cudadnn import CudaDnnDouble
from tests.conftest import bf16_round

pytestmark = pytest.mark.gpu


class _Side:
    def __init__(self, dev, kind):
        self.kind, self.half = kind, kind == "bf16"
        self.dev = dev
        self.cuda = CudaDnnDouble(0) if kind == "double" else dev.cuda
        self.tol = {"float": 2e-6, "bf16": 1e-2, "double": 1e-14}[kind]

    def put(self, a):
        """The handle of a's values and, in float64, the values as they are stored."""
        if self.kind == "double":
            return self.cuda.AllocMemory(np.asarray(a, np.float64).reshape(-1)), np.asarray(a, np.float64)
        a = np.asarray(a, np.float32)
        a = bf16_round(a) if self.half else a
        return self.dev.put(a, self.half), a.astype(np.float64)

    def zeros(self, n):
        return self.put(np.zeros(n))[0]

    def check(self, h, want, scale=1.0):
        if self.kind == "double":
            got = self.cuda.GetMemoryFloat(h, want.size).reshape(want.shape)
        else:
            got = self.dev.get(h, want.shape)
        assert np.abs(got - want).max() <= self.tol * scale * max(np.abs(want).max(), 1e-30)


@pytest.fixture(params=["float", "bf16", "double"])
def side(request, dev):
    s = _Side(dev, request.param)
    yield s
    if request.param == "double":
        s.cuda.Dispose()


@pytest.mark.parametrize("B,T,dim", [(2, 3, 1), (1, 5, 37), (2, 7, 256), (2, 66, 288), (1, 4, 768), (1, 3, 2048), (2, 2, 2052)])
def test_rms_norm_with_residual_and_its_gradient(side, B, T, dim):
    rng = np.random.default_rng(dim)
    rows, eps = B * T, 1e-5 if dim > 1 else 0.5   # a row of one value has no gradient but for eps
    (hx, x), (ha, a), (hdy, dy), (hres, res) = (side.put(rng.standard_normal((rows, dim))) for _ in range(4))
    hw, w = side.put(1 + 0.1 * rng.standard_normal(dim))
    ht, hy, hdx, hdw = side.zeros(x.size), side.zeros(x.size), side.zeros(x.size), side.put(np.full(dim, 7.0))[0]
    side.cuda.NormAddForward(0, rows, dim, hx, ha, ht, hw, hy, eps)
    side.check(ht, x + a)
    total = bf16_round((x + a).astype(np.float32)).astype(np.float64) if side.half else x + a
    side.check(hy, w * total / np.sqrt((total ** 2).mean(1, keepdims=True) + eps), 2)
    for add in (0, hres):
        side.cuda.RmsNormBackward(rows, dim, hx, hw, hdy, hdx, hdw, T, eps, add)
        r = 1 / np.sqrt((x ** 2).mean(1, keepdims=True) + eps)
        g = dy * w
        side.check(hdx, g * r - x * r ** 3 * (g * x).sum(1, keepdims=True) / dim + (res if add else 0), 4)
        side.check(hdw, (dy * x * r)[:T].sum(0), 4)


@pytest.mark.parametrize("rows,inner", [(3, 1), (6, 37), (5, 768), (2, 2048), (2, 2050)])
def test_layer_norm_with_residual(side, rows, inner):
    rng = np.random.default_rng(inner)
    eps = 1e-3
    (hx, x), (ha, a), (hdy, dy), (hres, res) = (side.put(rng.standard_normal((rows, inner))) for _ in range(4))
    ht, hy, hdx = (side.zeros(x.size) for _ in range(3))
    ln = side.cuda.CreateLayerNorm(0, x.size, rows, 1, inner, eps)
    side.cuda.NormAddForward(ln, 0, 0, hx, ha, ht, 0, hy)
    side.check(ht, x + a)
    total = bf16_round((x + a).astype(np.float32)).astype(np.float64) if side.half else x + a
    sd = np.sqrt(total.var(1, keepdims=True) + eps)
    y = (total - total.mean(1, keepdims=True)) / sd
    side.check(hy, y, 4)
    side.cuda.NormAddBackward(ln, hy, hdy, hdx, hres)
    div = np.repeat(sd, inner, 1)
    div.reshape(-1)[:rows] += eps   # the first entries of the row-expanded deviations grow by eps per backward call
    side.check(hdx, (dy - (y * (y * dy).mean(1, keepdims=True) + dy.mean(1, keepdims=True))) / div + res, 8)
    side.cuda.FreeLayerNorm(ln)


@pytest.mark.parametrize("B,T,H,hs,rope", [(1, 1, 1, 1, False), (2, 5, 3, 3, False), (2, 9, 2, 6, True), (3, 4, 5, 16, True), (1, 130, 2, 64, False)])
def test_gradient_of_the_head_layout(side, B, T, H, hs, rope):
    rng = np.random.default_rng(hs)
    parts = [side.put(rng.standard_normal((B, H, T, hs))) for _ in range(3)]
    C, hr = H * hs, 0
    hdx = side.zeros(B * T * 3 * C)
    if rope:
        hr = side.cuda.CreateRope(0, 0, B * T * C, B, T, H, hs, 10000.0)
    side.cuda.QkvHeadsGrad(B, T, H, hs, *[h for h, _ in parts], hdx, hr)
    vals = [v.copy() for _, v in parts]
    if rope:
        ang = np.arange(T)[:, None] / 10000.0 ** (np.arange(0, hs, 2) / hs)[None, :]
        c, s = np.cos(ang), np.sin(ang)
        for v in vals[:2]:
            re, im = v[..., 0::2].copy(), v[..., 1::2].copy()
            v[..., 0::2], v[..., 1::2] = re * c + im * s, im * c - re * s
    want = np.concatenate([v.transpose(0, 2, 1, 3).reshape(B * T, C) for v in vals], 1)
    side.check(hdx, want, 1e8 if rope and side.kind == "double" else 2)   # the tables come from float products
    if rope:
        side.cuda.FreeRope(hr)


@pytest.mark.parametrize("M,N,K", [(1, 1, 1), (4, 9, 3), (63, 20, 17), (255, 64, 64), (256, 72, 32), (1024, 68, 40), (1025, 66, 48), (2100, 96, 32)])
def test_inner_product_backward_and_heads_forward(side, M, N, K):
    rng = np.random.default_rng(M)
    (hx, x), (hdy, dy) = side.put(rng.standard_normal((M, K))), side.put(rng.standard_normal((M, N)))
    (hw, w), (hb, b) = side.put(rng.standard_normal((N, K))), side.put(rng.standard_normal(N))
    (hdw, dw), (hdb, db) = side.put(rng.standard_normal((N, K))), side.put(rng.standard_normal(N))
    hdx, dx = side.put(rng.standard_normal((M, K)))
    side.cuda.LinearBackward(M, N, K, hx, hw, hdy, hdw, hdb, hdx, True)
    side.check(hdw, dw + dy.T @ x, 2)
    side.check(hdb, db + dy.sum(0), 2)
    side.check(hdx, dx + dy @ w, 2)
    side.cuda.LinearBackward(M, N, K, hx, hw, hdy, hdw, 0, hdx)
    side.check(hdx, dy @ w, 2)
    T, heads = (M // 2 if M % 2 == 0 else M), (2 if N % 2 == 0 else 1)
    hy = side.zeros(M * N)
    side.cuda.LinearForward(M, N, K, hx, hw, hb, hy, T, heads)
    side.check(hy, (x @ w.T + b).reshape(M // T, T, heads, N // heads).transpose(0, 2, 1, 3), 2)


@pytest.mark.parametrize("n", [1, 7, 8, 4099])
def test_gated_silu_gradient(side, n):
    rng = np.random.default_rng(n)
    (ha, a), (hb, b), (hd, d) = (side.put(2 * rng.standard_normal(n)) for _ in range(3))
    hda, hdb = side.zeros(n), side.zeros(n)
    side.cuda.SwigluBackward(n, ha, hb, hd, hda, hdb)
    s = 1 / (1 + np.exp(-a))
    side.check(hda, d * b * s * (1 + a * (1 - s)), 4)
    side.check(hdb, d * a * s, 4)
