"""fp32 products with every value as two fp16 numbers (csrc/gemm_f32.hip, gemm_f32_split_kernel with PAIR): every tile, its edges, parts of a
contraction, and the values that two scaled fp16 numbers do not hold: beyond what the sample shows, far below the rest of their tile
or row, beside zeros."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# error over the sum of |a| |b|: 2^-23 of a value for either operand, 2^-22 for the product of the low parts, what the low parts may lose and
# three sums of 16 products, 2^-24 each, like a random walk
BOUND = lambda k: 2.0 ** -24 * (8 + 2 * np.sqrt(k))  # noqa: E731

SHAPES = [(1028, 4612, 580, 0, 1), (2052, 4100, 1028, 1, 1), (2052, 1544, 612, 2, 1), (516, 1540, 2052, 3, 2), (132, 132, 32004, 3, 28),
          (1027, 4613, 579, 0, 1), (2053, 4101, 1027, 1, 1), (2050, 1541, 611, 2, 1), (1030, 517, 4099, 3, 3), (1001, 770, 32003, 0, 9)]


def pair_tile(m, n, k):
    """The tile of the form with two fp16 numbers and the number of parts, None where another kernel takes the product."""
    from mycaffe_amd.cudadnn import load_library
    route = load_library().MCH_GemmFloatRoute(m, n, k, 1, 0) >> 16
    return (route % 16 - 1, route // 16) if route else None


def sample(rng, n):
    return np.unique(np.concatenate([[0, 1, n - 1, max(0, n - 4)], rng.integers(0, n, 60)]))


def product(dev, a, b, tA, tB, alpha=1.0, beta=0.0, c=None):
    (m, k), n = a.shape, b.shape[1]
    hc = dev.put(c) if c is not None else dev.zeros(m * n)
    dev.cuda.gemm(tA, tB, m, n, k, alpha, dev.put((a.T if tA else a).copy()), dev.put((b.T if tB else b).copy()), beta, hc)
    return dev.get(hc, (m, n))


def check(got, a, b, rows, cols, alpha=1.0, add=0.0):
    a, b = a[rows].astype(np.float64), b[:, cols].astype(np.float64)
    err, scale = np.abs(got[np.ix_(rows, cols)] - alpha * (a @ b) - add), np.abs(alpha) * (np.abs(a) @ np.abs(b))
    assert (err <= BOUND(a.shape[1]) * scale + 2.0 ** -23 * np.abs(add) + a.shape[1] * 2.0 ** -149).all(), (err / scale).max()


@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k,shape,parts", SHAPES)
def test_edges(dev, m, n, k, shape, parts, tA, tB):
    assert pair_tile(m, n, k) == (shape, parts)
    rng = np.random.default_rng(m + n + k)
    a, b, c = (rng.standard_normal(s, dtype=np.float32) for s in ((m, k), (k, n), (m, n)))
    rows, cols = sample(rng, m), sample(rng, n)
    check(product(dev, a, b, tA, tB, -0.5, 1.0, c), a, b, rows, cols, -0.5, c[np.ix_(rows, cols)])


def test_error_is_not_above_that_of_fp32_sums(dev):
    rng = np.random.default_rng(3)
    for m, n, k in ((8192, 768, 384), (2048, 1536, 768), (1024, 2304, 3072), (512, 1024, 8192)):
        assert pair_tile(m, n, k)
        a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
        got, rows = product(dev, a, b, False, True), sample(rng, m)
        want = a[rows].astype(np.float64) @ b.astype(np.float64)
        chain = np.zeros((len(rows), n), np.float32)
        for i in range(k):      # one rounding per product
            chain += np.multiply.outer(a[rows, i], b[i])
        norm = lambda d: np.sqrt((d ** 2).sum())  # noqa: E731
        assert norm(got[rows] - want) <= 0.75 * norm(chain - want), k


# scales of a row that its tile's scale does not reach, values that the sample does not see, products that leave nothing but small
# ones, rows and columns of zeros, beside ordinary rows in the same tiles
@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k", [s[:3] for s in SHAPES])
def test_values_that_two_parts_do_not_hold(dev, m, n, k, tA, tB):
    rng = np.random.default_rng(m + k)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    p2 = lambda e: np.float32(2.0 ** e)  # noqa: E731
    for v, w in ((a, b.T), (b.T, a)):
        for row, e in ((2, -8), (3, -12), (40, -30), (41, -100), (70, 9), (71, 14), (72, 40)):
            v[row] *= p2(e)
        v[90], v[91, 5:] = 0, 0
        v[100, k // 3] = p2(20)             # far beyond the rest
        v[101, :k // 2] *= p2(30)           # a row of two scales, the large one against zeros
        w[110, :k // 2] = 0
        v[102, ::7] *= p2(-40)              # tiny values among ordinary ones, and alone against what is not zero
        w[112] = 0
        w[112, ::7] = 1
        v[120] = np.where(rng.random(k) < 0.97, 0, v[120])   # few values
    got = product(dev, a, b, tA, tB)
    special = np.array([2, 3, 40, 41, 70, 71, 72, 90, 91, 100, 101, 102, 110, 112, 120])
    for rows, cols in ((special, np.arange(n)), (np.arange(m), special), (sample(rng, m), sample(rng, n))):
        check(got, a, b, rows, cols)
    assert (got[90] == 0).all() and (got[:, 90] == 0).all()


@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False)])
@pytest.mark.parametrize("m,n,k", [SHAPES[0][:3], SHAPES[7][:3]])
def test_infinities_and_nan(dev, m, n, k, tA, tB):
    rng = np.random.default_rng(6)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    a[7, k - 1], a[m - 1, 0], b[k - 1, n - 1], b[0, 3] = np.inf, np.nan, -np.inf, np.inf
    got = product(dev, a, b, tA, tB)
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    check(got, a, b, np.delete(np.arange(m), [7, m - 1])[::50], np.delete(np.arange(n), [3, n - 1])[::50])
