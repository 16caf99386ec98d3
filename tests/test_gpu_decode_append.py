"""Decode attention that rotates and appends in its own launch (csrc/attn_decode.hip, attn_decode_kernel with APPEND): one split and several,
the new position at the ends of a split, lanes past the row, cache layouts, and the calls that stay with two launches."""
import numpy as np
import pytest

from oracle import attention_ref as R

pytestmark = pytest.mark.gpu


def round_bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).view(np.float32)


def run(dev, B, H, kvH, L, S, hs, half, rope=True, merged=False, yOnQ=False):
    rng = np.random.default_rng(B * H + L + hs)
    cut = round_bf16 if half else lambda a: a
    q, kn, vn = (cut(rng.standard_normal((B, n, hs), dtype=np.float32)) for n in (H, kvH, kvH))
    # (B, kvH, S, hs) in memory, or (B, S, kvH, hs)
    kc, vc = (cut(rng.standard_normal((B, S, kvH, hs) if merged else (B, kvH, S, hs), dtype=np.float32)) for _ in range(2))
    put = lambda a: dev.cuda.AllocMemory(a, bHalfSize=half)  # noqa: E731
    hq, hkn, hvn, hk, hv = put(q), put(kn), put(vn), put(kc), put(vc)
    hy = hq if yOnQ else put(np.zeros_like(q))
    hr = dev.cuda.CreateRope(0, 0, B * H * hs, B, S, H, hs, 10000.0) if rope else 0
    sH, sT = (hs, kvH * hs) if merged else (S * hs, hs)
    dev.cuda.AttnDecodeForward(B, H, kvH, hs, L, hq, hk, hv, hy, kvH * S * hs, sH, sT, 0.0, hr, hkn, hvn)

    def get(h, a):
        f = dev.zeros(a.size)
        dev.cuda.copy(a.size, h, f)
        return dev.get(f, a.shape)

    cos, sin = (t.astype(np.float64) for t in R.rope_tables(S, hs)) if rope else (np.ones((S, hs // 2)), np.zeros((S, hs // 2)))

    def rot(x):
        o = x.astype(np.float64)
        o[..., 0::2], o[..., 1::2] = x[..., 0::2] * cos[L - 1] - x[..., 1::2] * sin[L - 1], x[..., 0::2] * sin[L - 1] + x[..., 1::2] * cos[L - 1]
        return cut(o.astype(np.float32))

    heads = lambda c: c.transpose(0, 2, 1, 3) if merged else c  # noqa: E731
    heads(vc)[:, :, L - 1] = vn
    # of a pair of up to sqrt(2) max: fp32 angles of up to L (two roundings of each, and of the products), then the storage type's rounding
    rel = np.sqrt(2) * ((2 * L + 4) * 2.0 ** -24 + (2.0 ** -8 if half else 0))
    qr = rot(q)
    if not yOnQ:
        assert np.abs(get(hq, q) - qr).max() <= rel * np.abs(q).max()
        qr = get(hq, q)
    newKey, got = get(hkn, kn), get(hk, kc)
    assert np.abs(newKey - rot(kn)).max() <= rel * np.abs(kn).max()
    heads(kc)[:, :, L - 1] = newKey
    assert np.array_equal(got, kc) and np.array_equal(get(hv, vc), vc)
    rep = lambda c: np.repeat(heads(c)[:, :, :L], H // kvH, axis=1)  # noqa: E731
    want = R.kv_cache_attention(qr, rep(kc), rep(vc), np.float64)
    # fp32 sums of hs and L terms, the result's rounding; on top of q the reference's own rotation of it is off by rel
    assert np.abs(get(hy, q) - want).max() <= ((2.0 ** -8 if half else 0) + 2.0 ** -24 * (hs + L) + (4 * rel if yOnQ else 0)) * np.abs(vc).max()
    if hr:
        dev.cuda.FreeRope(hr)


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("B,H,L,S,hs", [
    (1, 1, 1, 4, 64), (2, 4, 40, 64, 64), (1, 2, 129, 200, 64), (1, 2, 128, 200, 128), (3, 5, 65, 70, 128), (1, 2, 2000, 2048, 128), (1, 2, 1025, 1100, 64),
    (64, 8, 33, 40, 8), (2, 3, 50, 51, 24), (1, 1, 700, 700, 256), (8, 32, 300, 300, 128)])
def test_append(dev, B, H, L, S, hs, half):
    run(dev, B, H, H, L, S, hs, half)


@pytest.mark.parametrize("half", [False, True])
def test_layouts_and_two_launches(dev, half):
    run(dev, 2, 4, 4, 77, 90, 64, half, merged=True)
    run(dev, 2, 4, 4, 77, 90, 64, half, rope=False)
    run(dev, 2, 6, 2, 77, 90, 64, half)               # a key head for three heads
    run(dev, 2, 4, 4, 77, 90, 64, half, yOnQ=True)    # the result on top of q
    run(dev, 2, 3, 3, 30, 40, 18, half)               # rows without whole 16-byte pieces
