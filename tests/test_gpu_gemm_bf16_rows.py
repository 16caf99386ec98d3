"""16-bit products of up to 32 rows (csrc/gemm_bf16.hip, gemm_b16_rows_kernel): both row counts of a tile, columns that do not fill one,
contractions around one stage of 128 k and around what the wavefronts share, the epilogues, a result on top of an operand."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def round_bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).view(np.float32)


def put(dev, a):
    return dev.cuda.AllocMemory(round_bf16(a), bHalfSize=True)


def get(dev, h, shape):
    f = dev.zeros(int(np.prod(shape)))
    dev.cuda.copy(int(np.prod(shape)), h, f)
    return dev.get(f, shape)


def draw(*shapes):
    rng = np.random.default_rng(sum(sum(s) for s in shapes))
    return [round_bf16(rng.standard_normal(s, dtype=np.float32)) for s in shapes]


def close(got, want, scale, k):
    # one rounding to 16 bits, and of the fp32 sums one per product and wavefront at most
    assert (np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -24 * (k / 32 + 24) * scale).all()


@pytest.mark.parametrize("m", [1, 15, 16, 17, 32])
@pytest.mark.parametrize("n,k", [(1, 8), (16, 128), (17, 136), (40, 1048), (8, 2176), (4096, 264), (4100, 512), (8200, 520), (12290, 256), (24, 4096), (16, 8200)])
def test_edges(dev, m, n, k):
    a, b, c = draw((m, k), (n, k), (m, n))
    ha, hb, hc = put(dev, a), put(dev, b), put(dev, c)
    want, scale = a.astype(np.float64) @ b.T.astype(np.float64), np.abs(a.astype(np.float64)) @ np.abs(b.T.astype(np.float64))
    dev.cuda.gemm(False, True, m, n, k, -0.5, ha, hb, 1.0, hc)
    close(get(dev, hc, (m, n)), c - 0.5 * want, scale + np.abs(c), k)
    dev.cuda.LinearForward(m, n, k, ha, hb, 0, hc)
    close(get(dev, hc, (m, n)), want, scale, k)


@pytest.mark.parametrize("B,T,H,hs,rope", [(8, 1, 32, 128, False), (3, 7, 5, 16, True), (2, 16, 6, 20, True), (1, 1, 2, 4, False)])
def test_into_heads(dev, B, T, H, hs, rope):
    from oracle import attention_ref as R
    C = H * hs
    x, w, b = draw((B * T, C), (3 * C, C), (3 * C,))
    hq = [dev.cuda.AllocMemory(B * T * C, bHalfSize=True) for _ in range(3)]
    hr = dev.cuda.CreateRope(0, 0, B * T * C, B, T, H, hs, 10000.0) if rope else 0
    dev.cuda.QkvProjHeads(B, T, H, hs, put(dev, x), put(dev, w), put(dev, b), *hq, hr)
    ref = x.astype(np.float64) @ w.T.astype(np.float64) + b
    for i, h in enumerate(hq):
        third = ref.reshape(B, T, 3, H, hs)[:, :, i]
        want = R.rope_forward(third, T, H, hs, dtype=np.float64).reshape(B, T, H, hs) if rope and i < 2 else third
        # rounded to 16 bits before and after the rotation, which adds up two of them
        assert np.abs(get(dev, h, (B, H, T, hs)).transpose(0, 2, 1, 3) - want).max() <= (3 if rope else 1) * 2.0 ** -8 * np.abs(ref).max()
    if hr:
        dev.cuda.FreeRope(hr)


def test_infinities_and_nan(dev):
    m, n, k = 9, 40, 264
    a, b = draw((m, k), (n, k))
    a[5, 259], a[4, 0], a[8, 130] = np.inf, np.nan, -np.inf
    hc = put(dev, np.zeros((m, n), np.float32))
    dev.cuda.gemm(False, True, m, n, k, 1.0, put(dev, a), put(dev, b), 0.0, hc)
    got = get(dev, hc, (m, n))
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.T.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[[5, 8]], want[[5, 8]])
    rest = [i for i in range(m) if i not in (4, 5, 8)]
    close(got[rest], want[rest], np.abs(a[rest].astype(np.float64)) @ np.abs(b.T.astype(np.float64)), k)


def test_a_result_on_its_operand(dev):
    # one tile of columns: the tiles read all they need before they write, as before
    a, b = draw((8, 64), (64, 64))
    ha = put(dev, a)
    dev.cuda.gemm(False, True, 8, 64, 64, 1.0, ha, put(dev, b), 0.0, ha)
    want = a.astype(np.float64) @ b.T.astype(np.float64)
    close(get(dev, ha, (8, 64)), want, np.abs(a.astype(np.float64)) @ np.abs(b.T.astype(np.float64)), 64)
