"""Softmax rows of any length (quads or single elements in the lanes of one wavefront, one workgroup for a vocabulary), and the
causal chain whose zeros shorten the products and the gradient pass, at lengths that are no multiple of anything."""
import numpy as np
import pytest

from tests.conftest import bf16_round

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("log", [False, True])
@pytest.mark.parametrize("length", [1, 3, 37, 255, 257, 1023, 2047, 2048, 2049, 4100, 8193, 20002, 32768, 32769])
def test_softmax_forward_and_gradient(dev, length, log, half):
    rng = np.random.default_rng(length)
    rows = 5
    x, g = (rng.standard_normal((rows, length)).astype(np.float32) * 2 for _ in range(2))
    if half:
        x, g = bf16_round(x), bf16_round(g)
    hx, hg, hy, hd = dev.put(x, half), dev.put(g, half), dev.zeros(x.size, half), dev.zeros(x.size, half)
    hc, d = dev.cuda.CreateCuDNN(), dev.cuda.CreateTensorDesc()
    dev.cuda.SetTensorDesc(d, rows, length, 1, 1, half)
    dev.cuda.SoftmaxForward(hc, 2 if log else 1, 0, 1.0, d, hx, 0.0, d, hy)
    y = dev.get(hy, x.shape)
    e = x.astype(np.float64) - x.max(1, keepdims=True)
    ref = e - np.log(np.exp(e).sum(1, keepdims=True)) if log else np.exp(e) / np.exp(e).sum(1, keepdims=True)
    tol = 1e-2 if half else 2e-6
    assert np.abs(y - ref).max() <= tol * np.abs(ref).max() + 1e-30
    dev.cuda.SoftmaxBackward(hc, 2 if log else 1, 0, 1.0, d, hy, d, hg, 0.0, d, hd)
    y64, g64 = y.astype(np.float64), g.astype(np.float64)
    want = g64 - np.exp(y64) * g64.sum(1, keepdims=True) if log else (g64 - (g64 * y64).sum(1, keepdims=True)) * y64
    assert np.abs(dev.get(hd, x.shape) - want).max() <= (1e-2 if half else 1e-5) * max(np.abs(want).max(), 1e-30) + 1e-7


@pytest.mark.parametrize("B,T,C,H", [(2, 37, 48, 3), (1, 130, 64, 4), (2, 300, 128, 2)])
def test_explicit_chain_equals_the_attention_handle(dev, B, T, C, H):
    from mycaffe_amd.layers import Blob, CausalSelfAttentionLayer
    rng = np.random.default_rng(T)
    x = rng.standard_normal((B, T, C)).astype(np.float32)
    w = [rng.standard_normal(s).astype(np.float32) * 0.2 for s in ((3 * C, C), (3 * C,), (C, C), (C,))]
    dy = rng.standard_normal((B, T, C)).astype(np.float32)
    out = []
    for sdpa in (False, True):
        layer = CausalSelfAttentionLayer(dev.cuda, H, C, T, True, sdpa, training=True)
        bx, top = Blob(dev.cuda, x.shape), Blob(dev.cuda, x.shape)
        bx.mutable_cpu_data = x
        layer.Setup(bx, *w)
        for _ in range(2):   # the second pass finds the blobs of the first
            layer.Forward(bx, top)
            top.mutable_cpu_diff = dy
            layer.Backward(top, bx)
        out.append([top.mutable_cpu_data, bx.mutable_cpu_diff] + [b.mutable_cpu_diff for b in layer.c_attn.blobs + layer.c_proj.blobs])
    for a, b in zip(*out):
        assert np.abs(a - b).max() <= 2e-5 * np.abs(b).max()


@pytest.mark.parametrize("length", [1, 37, 64, 255, 1024, 2047, 2048, 2049, 4100, 32769])
def test_log_softmax_gradient_keeps_single_precision(dev, length):
    """dx = g - exp(y) sum(g) with a gradient of one value per row, the last: everywhere else dx = -exp(y), off by no more than
    the exponential (1 ulp) and its product with the sum, which is exactly 1 (2^-24 each way)."""
    rng = np.random.default_rng(length)
    y, g = -rng.uniform(0, 40, (3, length)).astype(np.float32), np.zeros((3, length), np.float32)
    g[:, -1] = 1.0
    hd, hc, d = dev.zeros(y.size), dev.cuda.CreateCuDNN(), dev.cuda.CreateTensorDesc()
    dev.cuda.SetTensorDesc(d, 3, length, 1, 1, False)
    dev.cuda.SoftmaxBackward(hc, 2, 0, 1.0, d, dev.put(y), d, dev.put(g), 0.0, d, hd)
    want = -np.exp(y[:, :-1].astype(np.float64))
    assert (np.abs(dev.get(hd, y.shape)[:, :-1] - want) <= 4 * 2.0 ** -24 * np.abs(want)).all()


@pytest.mark.parametrize("outer,T,hs,at", [(32, 512, 64, (5, 500, 9)), (3, 1023, 63, (-1, -1, -1))])   # the second: no whole quads, last value
@pytest.mark.parametrize("where", ["none", "dy above the diagonal", "dy on the diagonal", "v", "k", "q", "weights"])
def test_infinities_and_nan_spread_through_the_causal_zeros(dev, where, outer, T, hs, at):
    """0 x inf: a masked weight or its gradient is an exact zero, and still carries an infinity or a NaN of what it is multiplied by
    (sizes at which the products stop at the diagonal while everything is finite)."""
    cuda, rng = dev.cuda, np.random.default_rng(3)
    sc, dy = (rng.standard_normal((outer, T, T)).astype(np.float32) for _ in range(2))
    q, k, v = (rng.standard_normal((outer, T, hs)).astype(np.float32) for _ in range(3))
    if where == "dy above the diagonal":
        dy[2, 100, 400] = np.inf
    elif where == "dy on the diagonal":
        dy[2, 100, 100] = np.nan
    elif where in "qkv":
        {"q": q, "k": k, "v": v}[where][(at[0], 17, at[2]) if where == "q" else at] = -np.inf
    hp, hs_, hm, hd = dev.zeros(sc.size), dev.put(sc), dev.put(np.tril(np.ones((T, T), np.float32))), dev.zeros(sc.size)
    hc, d = cuda.CreateCuDNN(), cuda.CreateTensorDesc()
    cuda.SetTensorDesc(d, outer * T, T, 1, 1, False)
    cuda.scal(sc.size, 0.125, hs_)
    cuda.mask(sc.size, T * T, 0.0, -1e9, hs_, hm, hs_)
    cuda.SoftmaxForward(hc, 1, 0, 1.0, d, hs_, 0.0, d, hp)
    if where == "weights":
        cuda.set(1, hp, np.inf, 2 * T * T + 50 * T + 300)
    hout = dev.zeros(q.size)
    got, want = [], []
    with np.errstate(all="ignore"):
        masked = np.where(np.tril(np.ones((T, T))) == 0, -np.inf, sc.astype(np.float64) * 0.125)
        p = np.exp(masked - masked.max(-1, keepdims=True))
        p /= p.sum(-1, keepdims=True)
        if where == "weights":
            p[2, 50, 300] = np.inf
        ds = (dy.astype(np.float64) - (dy * p).sum(-1, keepdims=True)) * p
        for h, m, o, tA in ((hp, p, v, False), (hp, p, v, True), (hd, ds, k, False), (hd, ds, q, True)):
            if h == hd and len(got) == 2:
                cuda.SoftmaxBackward(hc, 1, 0, 1.0, d, hp, d, dev.put(dy), 0.0, d, hd)
                got.append(dev.get(hd, sc.shape))
                want.append(ds)
            cuda.matmul(outer, T, hs, T, h, dev.put(o), hout, 1.0, tA, False)
            got.append(dev.get(hout, o.shape))
            want.append((m.transpose(0, 2, 1) if tA else m) @ o.astype(np.float64))
    for i, (a, b) in enumerate(zip(got, want)):
        finite = np.isfinite(b)
        assert np.array_equal(np.isfinite(a), finite), (i, where)
        assert np.array_equal(np.isnan(a), np.isnan(b)), (i, where)
        assert np.abs(a[finite] - b[finite]).max() <= 2e-5 * np.abs(b[finite]).max(), (i, where)
