"""Values of fp32 products: what two fp32 numbers multiply to exactly comes out exactly, whichever kernel takes the product, and rows of
very different sizes, values far beyond or below the rest of their row, zeros, infinities and NaN."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LAYOUTS = [(False, True), (False, False), (True, False), (True, True)]
# large products in tiles of several sizes, their edges, contractions in parts, rows that 16-byte pieces do not divide
SIZES = [(1028, 4612, 580), (2052, 4100, 1028), (2052, 1544, 612), (516, 1540, 2052), (132, 132, 32004),
         (1027, 4613, 579), (2053, 4101, 1027), (2050, 1541, 611), (1030, 517, 4099), (1001, 770, 32003)]


def product(dev, a, b, tA, tB):
    (m, k), n = a.shape, b.shape[1]
    hc = dev.zeros(m * n)
    dev.cuda.gemm(tA, tB, m, n, k, 1.0, dev.put((a.T if tA else a).copy()), dev.put((b.T if tB else b).copy()), 0.0, hc)
    return dev.get(hc, (m, n))


def one_hot(where, width):
    s = np.zeros((len(where), width), np.float32)
    s[np.arange(len(where)), where] = 1
    return s


# a row of the one operand holds a single 1: the result is rows of the other, all 24 bits of them
@pytest.mark.parametrize("tA,tB", LAYOUTS)
@pytest.mark.parametrize("m,n,k", SIZES)
def test_selected_rows(dev, m, n, k, tA, tB):
    rng = np.random.default_rng(m + n + k)
    rows, cols = rng.integers(0, k, m), rng.integers(0, k, n)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    assert np.array_equal(product(dev, one_hot(rows, k), b, tA, tB), b[rows])
    assert np.array_equal(product(dev, a, one_hot(cols, k).T, tA, tB), a[:, cols])


# whole numbers of twelve bits, two a column, so that every sum is below 2^24
@pytest.mark.parametrize("tA,tB", LAYOUTS)
@pytest.mark.parametrize("m,n,k", SIZES)
def test_whole_numbers(dev, m, n, k, tA, tB):
    rng = np.random.default_rng(m + n + k)
    a, b = rng.integers(-2800, 2801, (m, k)).astype(np.float32), np.zeros((k, n), np.float32)
    at = np.stack([rng.integers(0, k // 2, n), rng.integers(k // 2, k, n)])
    b[at, np.arange(n)] = rng.integers(-2800, 2801, at.shape)
    want = (a[:, at[0]].astype(np.int64) * b[at[0], np.arange(n)].astype(np.int64) + a[:, at[1]].astype(np.int64) * b[at[1], np.arange(n)].astype(np.int64))
    assert np.array_equal(product(dev, a, b, tA, tB), want.astype(np.float32))


# gradients of an inner product whose incoming gradient names one output a row
@pytest.mark.parametrize("m,n,k", [(1500, 4096, 1024), (2052, 2052, 260), (1000, 8000, 772)])
def test_gradients_of_one_output_a_row(dev, m, n, k):
    rng = np.random.default_rng(n)
    x, w = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((n, k), dtype=np.float32)
    at = rng.permutation(n)[:m]
    h = [dev.put(v) for v in (x, w, one_hot(at, n), np.zeros((n, k)), np.zeros(n), np.zeros((m, k)))]
    dev.cuda.LinearBackward(m, n, k, *h)
    dw, db = np.zeros((n, k), np.float32), np.zeros(n, np.float32)
    dw[at], db[at] = x, 1
    assert np.array_equal(dev.get(h[3], (n, k)), dw) and np.array_equal(dev.get(h[4], (n,)), db) and np.array_equal(dev.get(h[5], (m, k)), w[at])


@pytest.mark.parametrize("B,T,H,hs", [(3, 700, 12, 64), (4, 2048, 3, 64), (1, 2044, 6, 48)])
def test_selected_rows_into_heads(dev, B, T, H, hs):
    C, rng = H * hs, np.random.default_rng(T)
    w, at = rng.standard_normal((3 * C, C), dtype=np.float32), rng.integers(0, C, B * T)
    hq = [dev.zeros(B * T * C) for _ in range(3)]
    dev.cuda.QkvProjHeads(B, T, H, hs, dev.put(one_hot(at, C)), dev.put(w), dev.put(np.zeros(3 * C)), *hq, 0)
    want = w.T[at].reshape(B, T, 3, H, hs)
    for i, h in enumerate(hq):
        assert np.array_equal(dev.get(h, (B, H, T, hs)).transpose(0, 2, 1, 3), want[:, :, i])


def check(got, a, b, rows, cols, lone=()):
    a, b = a[rows].astype(np.float64), b[:, cols].astype(np.float64)
    k = a.shape[1]
    # error over the sum of |a| |b|: a rounding of 2^-24 for at most every product and, of three parts a value, 6 sums of each 16, adding up
    # like a random walk, and what parts leave out (2^-25); results that end among the denormals.  Where one product is all there is of a
    # sum (`lone`), everything that comes after it is cut off at the same place: a last place (2^-23) for each of at most k / 2 partial sums.
    one = np.isin(rows, lone)[:, None] | np.isin(cols, lone)[None]
    scale = np.abs(a) @ np.abs(b)
    assert (np.abs(got[np.ix_(rows, cols)] - a @ b) <= 2.0 ** -24 * np.where(one, 2 + k, 2 + np.sqrt(k)) * scale + k * 2.0 ** -149).all()


def sample(rng, n):
    return np.unique(np.concatenate([[0, 1, n - 1, max(0, n - 4)], rng.integers(0, n, 60)]))


# scales of a row far from those of its tile, single values far beyond their row, products that leave nothing but small ones, rows and
# columns of zeros, beside ordinary rows in the same tiles
@pytest.mark.parametrize("tA,tB", LAYOUTS)
@pytest.mark.parametrize("m,n,k", SIZES)
def test_rows_of_many_scales(dev, m, n, k, tA, tB):
    rng = np.random.default_rng(m + k)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    p2 = lambda e: np.float32(2.0 ** e)  # noqa: E731
    for v, w in ((a, b.T), (b.T, a)):
        for row, e in ((2, -8), (3, -12), (40, -30), (41, -100), (70, 9), (71, 14), (72, 40)):
            v[row] *= p2(e)
        v[90], v[91, 5:] = 0, 0
        v[100, k // 3] = p2(20)             # far beyond the rest
        v[95, k // 2 + 1::97] *= p2(3)      # a little beyond it, beside tiny ones
        v[95, ::3] *= p2(-20)
        v[101, :k // 2] *= p2(30)           # a row of two scales, the large one against zeros
        w[110, :k // 2] = 0
        v[102, ::7] *= p2(-40)              # tiny values among ordinary ones, and alone against what is not zero
        w[112] = 0
        w[112, ::7] = 1
        v[120] = np.where(rng.random(k) < 0.97, 0, v[120])   # few values
    got = product(dev, a, b, tA, tB)
    special = np.array([2, 3, 40, 41, 70, 71, 72, 90, 91, 95, 100, 101, 102, 110, 112, 120])
    for rows, cols in ((special, np.arange(n)), (np.arange(m), special), (sample(rng, m), sample(rng, n))):
        check(got, a, b, rows, cols, (100,))
    assert (got[90] == 0).all() and (got[:, 90] == 0).all()


@pytest.mark.parametrize("tA,tB", LAYOUTS)
@pytest.mark.parametrize("m,n,k", [SIZES[0], SIZES[7]])
def test_infinities_and_nan(dev, m, n, k, tA, tB):
    rng = np.random.default_rng(6)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    a[7, k - 1], a[m - 1, 0], b[k - 1, n - 1], b[0, 3] = np.inf, np.nan, -np.inf, np.inf
    got = product(dev, a, b, tA, tB)
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    check(got, a, b, np.delete(np.arange(m), [7, m - 1])[::50], np.delete(np.arange(n), [3, n - 1])[::50])
