"""Attention of head sizes that the matrix-core kernels pad (csrc/attn_prefill.hip, csrc/attn_backward.hip with PADDED): sizes around each
kernel's, every kind of mask, lengths around the tiles, what lies past a row."""
import numpy as np
import pytest

from oracle import attention_ref as R
from tests.conftest import BF16_RTOL, FP32_RTOL, bf16_round
from tests.test_gpu_attention_backward import _check, _fwd_bwd, _probs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("hs", [4, 8, 16, 24, 32, 40, 48, 56, 72, 96, 120])
@pytest.mark.parametrize("B,H,Tq,Tk", [(2, 3, 130, 130), (1, 2, 65, 200), (1, 1, 1, 1), (3, 2, 31, 33)])
def test_masks(dev, B, H, Tq, Tk, hs, half):
    rng = np.random.default_rng(hs + Tq)
    q, dy = (bf16_round(rng.standard_normal((B, H, Tq, hs)).astype(np.float32)) for _ in range(2))
    k, v = (bf16_round(rng.standard_normal((B, H, Tk, hs)).astype(np.float32)) for _ in range(2))
    tol = BF16_RTOL if half else FP32_RTOL
    keys = (rng.random((B, Tk)) < 0.7).astype(np.float32)
    keys[0, 0] = 1
    if B > 2:
        keys[2] = 0      # masked everywhere: uniform weights
    batch = (rng.random((B, Tq, Tk)) < 0.6).astype(np.float32)
    batch[:, :, 0] = 1
    for mask, kind in ([(R.causal_mask(Tq), 0)] if Tq == Tk else []) + [(None, 0), (keys, 1), (batch, 2)]:
        _check(_fwd_bwd(dev, q, k, v, dy, mask, kind, half), q, k, v, dy, mask, kind, tol, "kind %d" % kind)


def test_infinite_neighbours(dev):
    # a row is padded with zeros, not with what lies behind it: -inf in a key keeps its weight at zero, and its row's neighbours unharmed
    rng = np.random.default_rng(3)
    q, k, v = (np.abs(rng.standard_normal((1, 1, 64, 16))).astype(np.float32) for _ in range(3))
    k[0, 0, 20, 3] = -np.inf
    hc, ha = dev.cuda.CreateCuDNN(), dev.cuda.CreateAttn()
    dev.cuda.SetAttn(hc, ha, 0, False, 1, 64, 1, 16, 0.0)
    hy = dev.zeros(q.size)
    dev.cuda.AttnScaledDotProductForward(hc, ha, 64, dev.put(q), dev.put(k), dev.put(v), 0, hy, 0)
    keep = np.delete(np.arange(64), 20)
    want = R.softmax_lastaxis(q.astype(np.float64) @ k[:, :, keep].swapaxes(-1, -2) / 4, np.float64) @ v[:, :, keep]
    assert np.abs(dev.get(hy, q.shape) - want).max() <= 1e-5 * np.abs(want).max()
    dev.cuda.FreeAttn(ha)
    dev.cuda.FreeCuDNN(hc)


# A causal row does not read what lies behind it: infinities and NaN in later keys and values leave the rows before them as they are, and the
# gradients of those rows.  hs 50 and 100: a kernel with a wavefront per row (16 bits), and none of a power of two.
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("hs", [8, 16, 48, 50, 72, 100])
@pytest.mark.parametrize("T,at", [(100, 20), (64, 63), (37, 33), (200, 130)])
@pytest.mark.parametrize("bad", [np.inf, -np.inf, np.nan])
def test_causal_rows_before_infinities(dev, T, at, hs, half, bad):
    rng = np.random.default_rng(hs + T)
    q, k, v, dy = (bf16_round(rng.standard_normal((1, 2, T, hs)).astype(np.float32)) for _ in range(4))
    mask, tol = R.causal_mask(T), BF16_RTOL if half else FP32_RTOL
    clean = _probs(q, k, mask, 0)
    want = [clean @ v.astype(np.float64), *R.attn_backward(q, k, v, clean, dy, np.float64)]
    k2, v2 = k.copy(), v.copy()
    k2[0, 0, at, 3], v2[0, 1, at, 5], v2[0, 1, at, hs - 1] = bad, bad, bad
    y, dq, dk, dv = _fwd_bwd(dev, q, k2, v2, dy, mask, 0, half)
    for got, exp in ((y, want[0]), (dq, want[1])):
        assert np.abs(got[:, :, :at] - exp[:, :, :at]).max() <= tol * np.abs(exp).max()
    # a value past its row's weight: that dimension of the rows from it on, no other
    others = np.setdiff1d(np.arange(hs), [5, hs - 1])
    assert np.abs(y[0, 1][:, others] - want[0][0, 1][:, others]).max() <= tol * np.abs(want[0]).max()
    assert np.array_equal(y[0, 1, at:, [5, hs - 1]], np.full((2, T - at), bad, np.float32), equal_nan=True)
    # the weights do not depend on values
    assert np.abs(dv[0, 1] - want[3][0, 1]).max() <= tol * np.abs(want[3]).max()


# the last key's row stands in for those past it, with weight zero: its own weight times infinity stays an infinity
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("hs", [16, 48, 72])
def test_infinity_in_the_last_value(dev, hs, half):
    rng = np.random.default_rng(hs)
    q, k, v = (bf16_round(rng.standard_normal((2, 2, 45, hs)).astype(np.float32)) for _ in range(3))
    v[0, 0, 44, 2], v[1, 1, 44, 7] = np.inf, -np.inf
    y = _fwd_bwd(dev, q, k, v, np.ones_like(q), None, 0, half)[0]
    with np.errstate(invalid="ignore"):
        want = _probs(q, k, None, 0) @ v.astype(np.float64)
    assert np.array_equal(np.isinf(y), np.isinf(want)) and np.array_equal(y[np.isinf(y)], want[np.isinf(want)].astype(np.float32))
    fine = np.isfinite(want)
    assert np.isfinite(y[fine]).all() and np.abs(y[fine] - want[fine]).max() <= (BF16_RTOL if half else FP32_RTOL) * np.abs(want[fine]).max()


# the same for the last query's row of the gradient
@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("hs", [16, 48, 72])
def test_infinity_in_the_last_gradient(dev, hs, half):
    rng = np.random.default_rng(hs)
    q, k, v, dy = (bf16_round(rng.standard_normal((1, 2, 45, hs)).astype(np.float32)) for _ in range(4))
    mask, dy2 = R.causal_mask(45), dy.copy()
    dy2[0, 1, 44, 2] = np.inf
    p = _probs(q, k, mask, 0)
    dv = _fwd_bwd(dev, q, k, v, dy2, mask, 0, half)[3]
    want = np.swapaxes(p, -1, -2) @ dy.astype(np.float64)
    want[0, 1, :, 2] = np.inf
    fine = np.isfinite(want)
    assert np.array_equal(dv[~fine], want[~fine].astype(np.float32)) and np.abs(dv[fine] - want[fine]).max() <= (BF16_RTOL if half else FP32_RTOL) * np.abs(want[fine]).max()


# 16-bit storage: weights and their gradients keep more than sixteen bits between the products, so that rounding the result is all that shows
@pytest.mark.parametrize("hs", [8, 16, 32, 48, 80, 96, 120])
@pytest.mark.parametrize("T,causal", [(64, True), (300, True), (300, False), (1000, True)])
def test_weights_keep_their_bits(dev, T, causal, hs):
    rng = np.random.default_rng(hs + T)
    q, k, v, dy = (bf16_round(rng.standard_normal((2, 2, T, hs)).astype(np.float32)) for _ in range(4))
    mask = R.causal_mask(T) if causal else None
    out = _fwd_bwd(dev, q, k, v, dy, mask, 0, True)
    q, k, v, dy = (a.astype(np.float64) for a in (q, k, v, dy))
    p = _probs(q, k, mask, 0)
    t = lambda a: np.swapaxes(a, -1, -2)  # noqa: E731
    ds = p * (dy @ t(v) - (out[0].astype(np.float64) * dy).sum(-1, keepdims=True)) / np.sqrt(hs)   # D from the result as it is stored
    norm = lambda a: np.sqrt((a ** 2).sum())  # noqa: E731
    for got, want in zip(out, (p @ v, ds @ k, t(ds) @ q, t(p) @ dy)):
        rounding = norm(bf16_round(want.astype(np.float32)) - want)
        # two roundings of 2^-17 and fp32 sums beside one of 2^-9: 1.0001; a weight rounded to 16 bits adds its own 2^-9 (1.2 - 1.4)
        assert norm(got - want) <= 1.002 * rounding
