"""The 16-bit GEMM kernel (csrc/gemm_bf16.hip) where it can go wrong: edges of each of its tiles (which of them a size goes to is asked of
the library), contractions that end inside a stage, every operand layout, contractions cut into parts, beta, and the bias and
head-layout epilogues."""
import numpy as np
import pytest

from tests.conftest import bf16_round

pytestmark = pytest.mark.gpu

# smallest, one past and one short of a tile, K of one chunk up to many stages, few tiles over a long K (parts), and sizes large
# enough for each of the wider tiles; multiples of 8 (what the kernel takes in every layout), the last two not in N or M
SHAPES = [(8, 8, 8), (64, 64, 64), (72, 56, 72), (128, 136, 200), (136, 264, 40), (200, 72, 2504), (768, 776, 8000), (2056, 1032, 264),
          (3080, 2312, 136), (8000, 776, 136), (8192, 1544, 72), (8008, 3080, 64), (5128, 4104, 72), (8136, 760, 776), (4104, 1144, 520), (100, 1001, 96), (1003, 136, 104)]


@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_gemm_edges(dev, m, n, k, tA, tB):
    rng = np.random.default_rng(m * 7 + n * 3 + k)
    a, b, c = (bf16_round(rng.standard_normal(s).astype(np.float32)) for s in ((m, k), (k, n), (m, n)))
    ha, hb = dev.put((a.T if tA else a).copy(), True), dev.put((b.T if tB else b).copy(), True)
    want = a @ b
    for alpha, beta in ((1.0, 0.0), (0.5, 1.0)):
        hc = dev.put(c, True)
        dev.cuda.gemm(tA, tB, m, n, k, alpha, ha, hb, beta, hc)
        ref = alpha * want + beta * c
        err = np.abs(dev.get(hc, (m, n)) - ref)
        assert (err <= 2.0 ** -8 * np.abs(ref) + 1e-5 * np.abs(ref).max()).all(), err.max()


def tile(m, n, k):
    """The number of the tile that the library takes for these sizes, and the parts of the contraction."""
    from mycaffe_amd.cudadnn import load_library
    route = load_library().MCH_GemmFloatRoute(m, n, k, 1, 8)
    return route // 4 % 16, route // 64


# every tile with edges, and those that parts of a contraction get
@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k,shape,parts", [(6152, 2312, 72, 0, 1), (3080, 4104, 136, 0, 1), (8008, 1032, 520, 1, 1), (4104, 4104, 520, 2, 1), (8008, 520, 520, 3, 1),
                                               (8008, 264, 72, 4, 1), (2056, 1032, 1544, 5, 1), (2056, 1032, 776, 6, 1), (8200, 72, 72, 7, 1), (72, 72, 136, 8, 1),
                                               (264, 6152, 72, 9, 1), (6152, 136, 4104, 3, 5), (8200, 72, 4104, 5, 3), (136, 6152, 4104, 6, 3), (72, 3080, 2056, 7, 5),
                                               (72, 72, 1032, 8, 4), (136, 3080, 4104, 9, 6)])
def test_every_tile(dev, m, n, k, shape, parts, tA, tB):
    assert tile(m, n, k) == (shape, parts)
    test_gemm_edges(dev, m, n, k, tA, tB)


@pytest.mark.parametrize("bias", [False, True])
@pytest.mark.parametrize("m,n,k", [(70, 66, 40), (5, 50, 704), (64, 64, 4096), (8000, 776, 136), (8008, 3080, 64), (300, 7, 72), (8136, 764, 776)])
def test_linear_forward_edges(dev, m, n, k, bias):
    rng = np.random.default_rng(n)
    x, w, b = (bf16_round(rng.standard_normal(s).astype(np.float32)) for s in ((m, k), (n, k), (n,)))
    hy = dev.zeros(m * n, True)
    dev.cuda.LinearForward(m, n, k, dev.put(x, True), dev.put(w, True), dev.put(b, True) if bias else 0, hy)
    ref = x @ w.T + (b if bias else 0)
    assert (np.abs(dev.get(hy, (m, n)) - ref) <= 2.0 ** -8 * np.abs(ref) + 1e-5 * np.abs(ref).max()).all()


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("B,T,H,hs", [(1, 1, 1, 8), (3, 37, 5, 24), (2, 65, 3, 40), (2, 700, 4, 96), (3, 33, 4, 6)])
def test_projection_into_heads_edges(dev, B, T, H, hs, rope, half):
    from oracle import attention_ref as R
    C = H * hs
    rng = np.random.default_rng(C + T)
    x, w, b = (bf16_round(rng.standard_normal(s).astype(np.float32)) for s in ((B, T, C), (3 * C, C), (3 * C,)))
    hq = [dev.zeros(B * T * C, half) for _ in range(3)]
    hr = dev.cuda.CreateRope(0, 0, B * T * C, B, T, H, hs, 10000.0) if rope else 0
    dev.cuda.QkvProjHeads(B, T, H, hs, dev.put(x, half), dev.put(w, half), dev.put(b, half), *hq, hr)
    ref = (x.astype(np.float64) @ w.T.astype(np.float64) + b).reshape(B, T, 3, H, hs)
    for i, h in enumerate(hq):
        want = R.rope_forward(ref[:, :, i], T, H, hs, dtype=np.float64).reshape(B, T, H, hs) if rope and i < 2 else ref[:, :, i]
        got = dev.get(h, (B, H, T, hs)).transpose(0, 2, 1, 3)
        assert np.abs(got - want).max() <= (2.0 ** -7 if half else 1e-4 if rope else 4e-6) * np.abs(ref).max()
    if hr:
        dev.cuda.FreeRope(hr)


# the ends in heads of every tile, with a rotation and without
@pytest.mark.parametrize("rope", [False, True])
@pytest.mark.parametrize("B,T,H,hs,shape", [(3, 2100, 11, 64, 0), (3, 2100, 11, 40, 1), (3, 2100, 5, 64, 2), (2, 1366, 8, 64, 3), (3, 2100, 3, 40, 4), (3, 171, 20, 64, 5),
                                            (3, 333, 8, 96, 6), (3, 1366, 3, 24, 7), (2, 65, 3, 40, 8), (3, 2100, 2, 24, 9)])
def test_projection_into_heads_of_every_tile(dev, B, T, H, hs, shape, rope):
    assert tile(B * T, 3 * H * hs, H * hs) == (shape, 1)
    test_projection_into_heads_edges(dev, B, T, H, hs, rope, True)
