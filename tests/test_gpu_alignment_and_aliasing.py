"""The kernels with wide accesses on operands that begin anywhere (whole shapes, odd first elements), the calls that may work in
place in place, and infinities and NaN through products and norms."""
import numpy as np
import pytest

from mycaffe_amd.cudadnn import CudaDnnError
from tests.conftest import bf16_round
from tests.test_gpu_block_fused import side  # noqa: F401  (the three storage types)

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k", [(128, 136, 200), (72, 264, 2504), (8136, 760, 72)])
def test_gemm_operands_that_begin_anywhere(dev, m, n, k, tA, tB, half):
    rng = np.random.default_rng(m + n)
    a, b, c = (bf16_round(rng.standard_normal(s).astype(np.float32)) for s in ((m, k), (k, n), (m, n)))
    want = 0.5 * (a.astype(np.float64) @ b) + c
    pad = np.full(8, 1e30, np.float32)
    buf = lambda x, t: dev.put(np.concatenate([pad, (x.T if t else x).reshape(-1)]), half)  # noqa: E731
    for oa, ob, oc in ((1, 0, 0), (0, 3, 0), (0, 0, 5), (4, 4, 4), (2, 6, 1)):   # first elements of an allocation of 8 more
        ha, hb = buf(a, tA), buf(b, tB)
        hc = dev.put(np.concatenate([pad[:oc], c.reshape(-1), pad[oc:]]), half)
        # the operand lies at 8; moved down so that it begins at its odd place
        for h, x, o in ((ha, a, oa), (hb, b, ob)):
            if o:
                dev.cuda.SetMemory(h, np.concatenate([pad[:o], (x.T if (tA if h == ha else tB) else x).reshape(-1), pad[o:]]))
        dev.cuda.gemm(tA, tB, m, n, k, 0.5, ha, hb, 1.0, hc, oa or 8, ob or 8, oc)
        got = dev.get(hc)
        err = np.abs(got[oc:oc + m * n].reshape(m, n) - want)
        assert (err <= (2.0 ** -8 if half else 2e-6 * max(1.0, np.sqrt(k) / 16)) * (np.abs(want) if half else np.abs(want).max()) + 1e-5).all()
        around = bf16_round(pad) if half else pad
        assert np.array_equal(got[:oc], around[:oc]) and np.array_equal(got[oc + m * n:], around[oc:])


class _Views:
    """Handles of memory pointers that begin `off` elements into an allocation of their own."""

    def __init__(self, side):  # noqa: F811
        self.side, self.views = side, []

    def put(self, a, off):
        h, values = self.side.put(np.concatenate([np.zeros(off), np.asarray(a).reshape(-1)]))
        if off:
            h = self.side.cuda.CreateMemoryPointer(h, off, a.size)
            self.views.append(h)
        return h, values[off:].reshape(np.shape(a))

    def close(self):
        for v in self.views:
            self.side.cuda.FreeMemoryPointer(v)


@pytest.fixture()
def views(side):  # noqa: F811
    v = _Views(side)
    yield v
    v.close()


@pytest.mark.parametrize("off", [1, 2, 4, 6])
def test_calls_of_a_block_on_operands_that_begin_anywhere(side, views, off):  # noqa: F811
    """Shapes that are whole in every vector width, one operand after the other (and all of them) off by some elements."""
    rng, cuda = np.random.default_rng(off), side.cuda
    B, T, H, hs, N = 2, 12, 2, 16, 64
    C, M = H * hs, B * T
    for which in list(range(6)) + ["all"]:
        o = lambda i: off if which in (i, "all") else 0  # noqa: E731
        # inner product and its gradient
        (hx, x), (hw, w), (hb, b), (hdy, dy) = (views.put(rng.standard_normal(s), o(i)) for i, s in enumerate(((M, C), (N, C), N, (M, N))))
        (hy, _), (hdx, _) = views.put(np.zeros((M, N)), o(4)), views.put(np.zeros((M, C)), o(5))
        hdw, hdb = views.put(np.zeros((N, C)), o(1))[0], views.put(np.zeros(N), o(2))[0]
        cuda.LinearForward(M, N, C, hx, hw, hb, hy)
        side.check(hy, x @ w.T + b, 2)
        cuda.LinearForward(M, N, C, hx, hw, hb, hy, T, 4)
        side.check(hy, (x @ w.T + b).reshape(B, T, 4, N // 4).transpose(0, 2, 1, 3), 2)
        cuda.LinearBackward(M, N, C, hx, hw, hdy, hdw, hdb, hdx)
        side.check(hdw, dy.T @ x, 2)
        side.check(hdb, dy.sum(0), 2)
        side.check(hdx, dy @ w, 2)
        # projection into heads, and the gradient of that layout
        hw3, w3 = views.put(rng.standard_normal((3 * C, C)), o(1))
        hb3, b3 = views.put(rng.standard_normal(3 * C), o(2))
        q = [views.put(np.zeros((B, H, T, hs)), o(3 + i))[0] for i in range(3)]
        cuda.QkvProjHeads(B, T, H, hs, hx, hw3, hb3, *q)
        want = (x @ w3.T + b3).reshape(B, T, 3, H, hs).transpose(2, 0, 3, 1, 4)
        for i in range(3):
            side.check(q[i], want[i], 2)
        parts = [views.put(rng.standard_normal((B, H, T, hs)), o(i)) for i in range(3)]
        hg, _ = views.put(np.zeros((M, 3 * C)), o(3))
        cuda.QkvHeadsGrad(B, T, H, hs, *[h for h, _ in parts], hg)
        side.check(hg, np.concatenate([v.transpose(0, 2, 1, 3).reshape(M, C) for _, v in parts], 1), 2)
        # norms with their residuals
        eps = 1e-3
        (ha, a), (hn, n), (hres, res) = views.put(rng.standard_normal((M, C)), o(1)), views.put(1 + rng.standard_normal(C), o(2)), views.put(rng.standard_normal((M, C)), o(3))
        ht, hy2 = views.put(np.zeros((M, C)), o(4))[0], views.put(np.zeros((M, C)), o(5))[0]
        total = bf16_round((x + a).astype(np.float32)).astype(np.float64) if side.half else x + a
        cuda.NormAddForward(0, M, C, hx, ha, ht, hn, hy2, eps)
        side.check(ht, x + a)
        r = 1 / np.sqrt((total ** 2).mean(1, keepdims=True) + eps)
        side.check(hy2, n * total * r, 4)
        hdw2 = views.put(np.zeros(C), o(5))[0]
        hg2, g2 = views.put(rng.standard_normal((M, C)), o(2))
        cuda.RmsNormBackward(M, C, hx, hn, hg2, hdx, hdw2, M, eps, hres)
        r = 1 / np.sqrt((x ** 2).mean(1, keepdims=True) + eps)
        gw = g2 * n
        side.check(hdx, gw * r - x * r ** 3 * (gw * x).mean(1, keepdims=True) + res, 8)
        side.check(hdw2, (g2 * x * r).sum(0), 8)
        ln = cuda.CreateLayerNorm(0, M * C, M, 1, C, eps)
        cuda.NormAddForward(ln, 0, 0, hx, ha, ht, 0, hy2)
        sd = np.sqrt(total.var(1, keepdims=True) + eps)
        y = (total - total.mean(1, keepdims=True)) / sd
        side.check(hy2, y, 4)
        cuda.NormAddBackward(ln, hy2, hg2, hdx, hres)
        div = np.repeat(sd, C, 1)
        div.reshape(-1)[:M] += eps
        side.check(hdx, (g2 - (y * (y * g2).mean(1, keepdims=True) + g2.mean(1, keepdims=True))) / div + res, 8)
        cuda.FreeLayerNorm(ln)
        # gated SiLU
        hda, hdb2 = views.put(np.zeros((M, C)), o(4))[0], views.put(np.zeros((M, C)), o(5))[0]
        cuda.SwigluBackward(M * C, hx, ha, hg2, hda, hdb2)
        s = 1 / (1 + np.exp(-x))
        side.check(hda, g2 * a * s * (1 + x * (1 - s)), 4)
        side.check(hdb2, g2 * x * s, 4)


@pytest.mark.parametrize("inner", [37, 256, 2048, 2052])
@pytest.mark.parametrize("layer", [False, True])
def test_norms_with_residual_in_place(side, inner, layer):  # noqa: F811
    rng, cuda, rows, eps = np.random.default_rng(inner), side.cuda, 5, 1e-3
    (x0, a0, g0, r0), w0 = rng.standard_normal((4, rows, inner)), 1 + 0.1 * rng.standard_normal(inner)
    ln = cuda.CreateLayerNorm(0, rows * inner, rows, 1, inner, eps) if layer else 0
    for total_in, y_in in (("x", None), ("add", None), (None, "x"), (None, "add"), ("x", "add"), ("add", "x")):
        (hx, x), (ha, a), (hw, w) = side.put(x0), side.put(a0), side.put(w0)
        ht = {"x": hx, "add": ha, None: side.zeros(x.size)}[total_in]
        hy = {"x": hx, "add": ha, None: side.zeros(x.size)}[y_in]
        cuda.NormAddForward(ln, rows, inner, hx, ha, ht, 0 if layer else hw, hy, eps)
        total = bf16_round((x + a).astype(np.float32)).astype(np.float64) if side.half else x + a
        side.check(ht, x + a)
        if layer:
            side.check(hy, (total - total.mean(1, keepdims=True)) / np.sqrt(total.var(1, keepdims=True) + eps), 4)
        else:
            side.check(hy, w * total / np.sqrt((total ** 2).mean(1, keepdims=True) + eps), 4)
    with pytest.raises(CudaDnnError):    # total and y are two results
        cuda.NormAddForward(ln, rows, inner, hx, ha, ht, 0 if layer else hw, ht, eps)
    for into in ("y", "dy", "add"):
        (hx, x), (hg, g), (hr, r), (hw, w) = side.put(x0), side.put(g0), side.put(r0), side.put(w0)
        if layer:
            hy = side.zeros(x.size)
            cuda.NormAddForward(ln, rows, inner, hx, side.zeros(x.size), side.zeros(x.size), 0, hy, eps)
            sd = np.sqrt(x.var(1, keepdims=True) + eps)
            y = (x - x.mean(1, keepdims=True)) / sd
            y = bf16_round(y.astype(np.float32)).astype(np.float64) if side.half else y
            h = {"y": hy, "dy": hg, "add": hr}[into]
            cuda.NormAddBackward(ln, hy, hg, h, hr)
            div = np.repeat(sd, inner, 1)
            div.reshape(-1)[:rows] += eps
            side.check(h, (g - (y * (y * g).mean(1, keepdims=True) + g.mean(1, keepdims=True))) / div + r, 8)
        else:
            h = {"y": hx, "dy": hg, "add": hr}[into]
            cuda.RmsNormBackward(rows, inner, hx, hw, hg, h, 0, 0, eps, hr)
            s = 1 / np.sqrt((x ** 2).mean(1, keepdims=True) + eps)
            gw = g * w
            side.check(h, gw * s - x * s ** 3 * (gw * x).mean(1, keepdims=True) + r, 8)
            if into != "add":            # the weight gradient reads x and dy afterwards
                with pytest.raises(CudaDnnError):
                    cuda.RmsNormBackward(rows, inner, hx, hw, hg, h, side.zeros(inner), rows, eps, hr)
    if ln:
        cuda.FreeLayerNorm(ln)


@pytest.mark.parametrize("n", [8, 4099])
def test_gated_silu_gradient_in_place(side, n):  # noqa: F811
    rng, cuda = np.random.default_rng(n), side.cuda
    vals = rng.standard_normal((3, n))
    for da, db in (("a", "b"), ("b", "a"), ("dy", "a"), ("a", "dy"), ("dy", "b")):
        (ha, a), (hb, b), (hd, d) = (side.put(v) for v in vals)
        h = {"a": ha, "b": hb, "dy": hd}
        cuda.SwigluBackward(n, ha, hb, hd, h[da], h[db])
        s = 1 / (1 + np.exp(-a))
        side.check(h[da], d * b * s * (1 + a * (1 - s)), 4)
        side.check(h[db], d * a * s, 4)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("m,n,k", [(72, 264, 200), (136, 64, 4096), (8192, 2304, 256)])
def test_products_carry_infinities_and_nan(dev, m, n, k, half):
    """Chunks past the end of a tile or of the contraction are zeros that meet nothing: only rows and columns that hold one show it."""
    rng = np.random.default_rng(m)
    x, w, b = (rng.integers(1, 4, s).astype(np.float32) for s in ((m, k), (n, k), n))
    x[m - 1, k - 1], x[3, 0], w[n - 1, k - 1], b[5] = np.inf, np.nan, -np.inf, np.nan
    with np.errstate(invalid="ignore"):
        want = x.astype(np.float64) @ w.T.astype(np.float64) + b
        dwant = (x.T.astype(np.float64) @ x[:, :8].astype(np.float64)) if m < 1000 else None
    hx, hy = dev.put(x, half), dev.zeros(m * n, half)
    dev.cuda.LinearForward(m, n, k, hx, dev.put(w, half), dev.put(b, half), hy)
    got = dev.get(hy, (m, n))
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isposinf(got), np.isposinf(want))
    assert np.array_equal(np.isneginf(got), np.isneginf(want))
    ok = np.isfinite(want)
    assert (np.abs(got[ok] - want[ok]) <= (2.0 ** -8 if half else 0) * np.abs(want[ok])).all()
    if dwant is not None:
        hg = dev.zeros(k * 8, half)
        dev.cuda.gemm(True, False, k, 8, m, 1.0, hx, dev.put(x[:, :8].copy(), half), 0.0, hg)
        got = dev.get(hg, (k, 8))
        assert np.array_equal(np.isnan(got), np.isnan(dwant)) and np.array_equal(np.isinf(got), np.isinf(dwant))


@pytest.mark.parametrize("inner", [37, 256, 2052])
def test_a_row_of_a_norm_that_is_not_finite_stays_alone(side, inner):  # noqa: F811
    rng, cuda, rows, eps = np.random.default_rng(inner), side.cuda, 6, 1e-3
    x = rng.standard_normal((rows, inner))
    x[2, inner - 1], x[4, 0] = np.inf, np.nan
    (hx, x), (ha, a), (hw, w) = side.put(x), side.put(rng.standard_normal((rows, inner))), side.put(np.ones(inner))
    for ln in (0, cuda.CreateLayerNorm(0, rows * inner, rows, 1, inner, eps)):
        ht, hy = side.zeros(x.size), side.zeros(x.size)
        cuda.NormAddForward(ln, rows, inner, hx, ha, ht, 0 if ln else hw, hy, eps)
        got = (side.cuda.GetMemoryFloat(hy, x.size) if side.kind == "double" else side.dev.get(hy)).reshape(rows, inner)
        assert np.isfinite(got[[0, 1, 3, 5]]).all()
        assert np.isnan(got[2, inner - 1]) and np.isnan(got[4]).all()
        if ln:
            cuda.FreeLayerNorm(ln)
