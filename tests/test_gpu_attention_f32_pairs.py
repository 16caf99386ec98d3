"""fp32 attention whose rows are shared by two wavefronts (heads of at most 64): outputs and gradients against float64."""
import numpy as np
import pytest

from oracle import attention_ref as R

pytestmark = pytest.mark.gpu


def exact(q, k, v, dy, masked, scale):
    """y, dq, dk, dv in float64; `masked` (B,1,T,T) scores are filled, which weighs all keys of a row without any other alike."""
    q, k, v, dy = (x.astype(np.float64) for x in (q, k, v, dy))
    s = q @ k.swapaxes(-1, -2) * scale
    s = np.where(masked, R.MASKED, s)
    p = np.exp(s - s.max(-1, keepdims=True))
    p /= p.sum(-1, keepdims=True)
    dp = dy @ v.swapaxes(-1, -2)
    ds = p * (dp - (p * dp).sum(-1, keepdims=True))
    return p @ v, ds @ k * scale, ds.swapaxes(-1, -2) @ q * scale, p.swapaxes(-1, -2) @ dy


# one step of 32 and its edges, two steps (each wavefront's first), the edge of a 64-row workgroup, an odd number of steps
@pytest.mark.parametrize("T", [33, 63, 64, 65, 97, 160, 257])
@pytest.mark.parametrize("hs", [12, 32, 48, 64])
@pytest.mark.parametrize("kind", ["none", "causal", "key", "qk"])
def test_pairs_of_wavefronts(dev, kind, hs, T):
    c, B, H = dev.cuda, 2, 3
    rng = np.random.default_rng(T * 100 + hs)
    q, k, v, dy = (rng.standard_normal((B, H, T, hs)).astype(np.float32) for _ in range(4))
    mask = {"none": None, "causal": R.causal_mask(T),
            # the first sequence sees only keys of the second wavefront's steps, the second one none at all
            "key": np.stack([(np.arange(T) >= 32), np.zeros(T, bool)]).astype(np.float32),
            "qk": (rng.random((T, T)) < 0.5).astype(np.float32)}[kind]
    if kind == "qk":
        mask[5] = 0
        mask[7, :32], mask[9, 32:] = 0, 0
    masked = np.zeros((B, 1, T, T), bool)
    if mask is not None:
        masked |= (np.asarray(mask).reshape((B, 1, 1, T) if kind == "key" else (1, 1, T, T)) == 0)
    want = exact(q, k, v, dy, masked, 1 / np.sqrt(hs))
    h = [c.AllocMemory(x.ravel()) for x in (q, k, v, dy)]
    out = [c.AllocMemory(q.size) for _ in range(4)]
    hm = c.AllocMemory(np.asarray(mask, np.float32).ravel()) if mask is not None else 0
    hc, ha = c.CreateCuDNN(), c.CreateAttn()
    c.SetAttn(hc, ha, 0, True, B, T, H, hs, 0.0)
    c.AttnScaledDotProductForward(hc, ha, T, *h[:3], hm, out[0], 1 if kind == "key" else 0, None)
    c.AttnScaledDotProductBackward(hc, ha, h[0], out[1], h[1], out[2], h[2], out[3], hm, out[0], h[3])
    got = [np.asarray(c.GetMemoryFloat(o, q.size)).reshape(q.shape) for o in out]
    # scores of standard normal rows are sums of hs products with a rounding of 2^-24 each, |s| below 6; a weight's relative error is the
    # score's absolute one, and sums over up to T keys of values below 5 add T/2 roundings at most: 3e-5 of the largest value covers both
    for name, a, b in zip(("y", "dq", "dk", "dv"), got, want):
        assert np.isfinite(a).all(), name
        assert np.abs(a - b).max() <= 3e-5 * max(np.abs(b).max(), 1.0), name
    for x in (*h, *out, *([hm] if hm else [])):
        c.FreeMemory(x)
    c.FreeAttn(ha)


@pytest.mark.parametrize("hs", [48, 64])
def test_a_step_of_scores_at_minus_infinity(dev, hs):
    """keys 32 .. 63 score -inf for every row: the second wavefront's first step has no weight, its later ones have"""
    c, B, H, T = dev.cuda, 1, 2, 130
    rng = np.random.default_rng(hs)
    q, k, v = (rng.standard_normal((B, H, T, hs)).astype(np.float32) for _ in range(3))
    q[..., 0] = 1.0
    keep = np.r_[0:32, 64:T]
    want = exact(q, k[:, :, keep], v[:, :, keep], q, np.zeros((B, 1, T, len(keep)), bool), 1 / np.sqrt(hs))[0]
    k[:, :, 32:64, 0] = -np.inf
    h = [c.AllocMemory(x.ravel()) for x in (q, k, v)]
    y = c.AllocMemory(q.size)
    hc, ha = c.CreateCuDNN(), c.CreateAttn()
    c.SetAttn(hc, ha, 0, True, B, T, H, hs, 0.0)
    c.AttnScaledDotProductForward(hc, ha, T, *h, 0, y, 0, None)
    got = np.asarray(c.GetMemoryFloat(y, q.size)).reshape(q.shape)
    assert np.abs(got - want).max() <= 3e-5 * np.abs(want).max()
    for x in (*h, y):
        c.FreeMemory(x)
    c.FreeAttn(ha)


@pytest.mark.parametrize("kind", ["none", "causal", "key", "qk"])
@pytest.mark.parametrize("hs", [48, 64])
def test_every_score_at_minus_infinity(dev, hs, kind):
    """a softmax over scores of -inf alone has no weights: outputs and all gradients of that head are NaN, those of its neighbours are not"""
    c, B, H, T = dev.cuda, 1, 2, 130
    rng = np.random.default_rng(hs)
    q, k, v, dy = (rng.standard_normal((B, H, T, hs)).astype(np.float32) for _ in range(4))
    q[..., 0] = 1.0
    k[:, 0, :, 0] = -np.inf
    mask = {"none": None, "causal": R.causal_mask(T), "key": np.ones((B, T), np.float32), "qk": np.ones((T, T), np.float32)}[kind]
    masked = np.zeros((B, 1, T, T), bool) | (np.asarray(R.causal_mask(T)).reshape(1, 1, T, T) == 0) if kind == "causal" else np.zeros((B, 1, T, T), bool)
    want = exact(q[:, 1:], k[:, 1:], v[:, 1:], dy[:, 1:], masked, 1 / np.sqrt(hs))
    h = [c.AllocMemory(x.ravel()) for x in (q, k, v, dy)]
    out = [c.AllocMemory(q.size) for _ in range(4)]
    hm = c.AllocMemory(np.asarray(mask, np.float32).ravel()) if mask is not None else 0
    hc, ha = c.CreateCuDNN(), c.CreateAttn()
    c.SetAttn(hc, ha, 0, True, B, T, H, hs, 0.0)
    c.AttnScaledDotProductForward(hc, ha, T, *h[:3], hm, out[0], 1 if kind == "key" else 0, None)
    c.AttnScaledDotProductBackward(hc, ha, h[0], out[1], h[1], out[2], h[2], out[3], hm, out[0], h[3])
    for name, o, w in zip(("y", "dq", "dk", "dv"), out, want):
        got = np.asarray(c.GetMemoryFloat(o, q.size)).reshape(q.shape)
        assert np.isnan(got[:, 0]).all(), name
        assert np.abs(got[:, 1:] - w).max() <= 3e-5 * max(np.abs(w).max(), 1.0), name
    for x in (*h, *out, *([hm] if hm else [])):
        c.FreeMemory(x)
    c.FreeAttn(ha)


@pytest.mark.parametrize("training", [True, False])
@pytest.mark.parametrize("hs", [32, 64])
def test_one_order_of_a_rows_sums(dev, hs, training):
    """bOneWave: a sequence's outputs are the same bits alone, where several wavefronts would share its rows, and among many"""
    c, H, T, many = dev.cuda, 4, 130, 200
    rng = np.random.default_rng(hs)
    x = [rng.standard_normal((many, H, T, hs)).astype(np.float32) for _ in range(3)]
    outs = []
    for B in (1, many):
        h = [c.AllocMemory(a[:B].ravel()) for a in x]
        hm, y = c.AllocMemory(R.causal_mask(T).ravel()), c.AllocMemory(B * H * T * hs)
        hc, ha = c.CreateCuDNN(), c.CreateAttn()
        c.SetAttn(hc, ha, 0, training, B, T, H, hs, 0.0)
        c.AttnScaledDotProductForward(hc, ha, T, *h, hm, y, 0, bOneWave=True)
        outs.append(np.asarray(c.GetMemoryFloat(y, H * T * hs)))
        for m in (*h, hm, y):
            c.FreeMemory(m)
        c.FreeAttn(ha)
    assert np.array_equal(*outs)
