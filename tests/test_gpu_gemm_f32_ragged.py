"""fp32 products on the bf16 matrix cores whose operands are no whole aligned 16-byte chunks (csrc/gemm_f32.hip, gemm_f32_split_kernel, kTail):
every remainder of rows, columns and contraction, operands off their alignment, rows of one and two values, what lies past a row."""
import numpy as np
import pytest

from tests.test_gpu_gemm_f32_split import tile

pytestmark = pytest.mark.gpu

BOUND = lambda k: 2.0 ** -24 * (2 + np.sqrt(6 * k / 16))  # noqa: E731  (of the sum of |a| |b|: as for whole chunks)


def sample(rng, n):
    return np.unique(np.concatenate([[0, 1 % n, n - 1, max(0, n - 2), max(0, n - 3), max(0, n - 5)], rng.integers(0, n, 40)]))


def check(got, a, b, rows, cols, alpha=1.0, add=0.0):
    a, b = a[rows].astype(np.float64), b[:, cols].astype(np.float64)
    err = np.abs(got[np.ix_(rows, cols)] - alpha * (a @ b) - (add[np.ix_(rows, cols)] if np.ndim(add) else add))
    assert (err <= BOUND(a.shape[1]) * (abs(alpha) * (np.abs(a) @ np.abs(b)) + 1.0)).all(), err.max()


# every tile, parts; all remainders of four in each size
@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k,shape", [(2053, 4101, 69, 3), (2055, 2050, 162, 3), (517, 262, 4099, 5), (131, 133, 32001, 5), (4097, 3073, 65, 3), (1000, 3, 140001, 5),
                                         (2, 2049, 70000, 4), (1, 3000, 100003, 4), (4101, 3075, 293, 0), (3077, 3077, 291, 1), (1027, 4613, 579, 2),
                                         (2055, 1541, 303, 4), (2050, 1541, 611, 3), (2048, 2048, 1023, 3), (2049, 2048, 1024, 2),
                                         (1029, 1027, 611, None), (1024, 1024, 1023, None), (1025, 1024, 1024, None)])   # the last: gemm_f32_small_kernel
def test_remainders(dev, m, n, k, shape, tA, tB):
    assert tile(m, n, k) == shape
    rng = np.random.default_rng(m + n + k)
    a, b, c = (rng.standard_normal(s, dtype=np.float32) for s in ((m, k), (k, n), (m, n)))
    ha, hb, hc = dev.put((a.T if tA else a).copy()), dev.put((b.T if tB else b).copy()), dev.put(c)
    rows, cols = sample(rng, m), sample(rng, n)
    dev.cuda.gemm(tA, tB, m, n, k, -0.5, ha, hb, 1.0, hc)
    check(dev.get(hc, (m, n)), a, b, rows, cols, -0.5, c)


@pytest.mark.parametrize("tA,tB", [(False, True), (True, False)])
@pytest.mark.parametrize("m,n,k,shape", [(2100, 1030, 515, 5), (1024, 1030, 515, None)])
def test_offsets(dev, m, n, k, shape, tA, tB):
    assert tile(m, n, k) == shape
    rng = np.random.default_rng(5)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    for oa, ob, oc in ((1, 0, 0), (0, 3, 2), (2, 1, 1)):
        ha, hb = (dev.put(np.concatenate([np.full(o, np.nan, np.float32), x.ravel(), np.full(3, np.nan, np.float32)]))
                  for o, x in ((oa, a.T if tA else a), (ob, b.T if tB else b)))
        hc = dev.zeros(m * n + oc)
        dev.cuda.gemm(tA, tB, m, n, k, 1.0, ha, hb, 0.0, hc, oa, ob, oc)
        check(dev.get(hc, (m * n + oc,))[oc:].reshape(m, n), a, b, sample(rng, m), sample(rng, n))


@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False)])
@pytest.mark.parametrize("m,n,k,shape", [(3003, 1029, 303, 4), (1027, 1029, 303, None)])
def test_infinities_stay_in_their_rows(dev, m, n, k, shape, tA, tB):
    assert tile(m, n, k) == shape
    rng = np.random.default_rng(6)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    a[7, k - 1], a[m - 1, 0], b[k - 1, 1028], b[0, 3] = np.inf, np.nan, -np.inf, np.inf
    hc = dev.zeros(m * n)
    dev.cuda.gemm(tA, tB, m, n, k, 1.0, dev.put((a.T if tA else a).copy()), dev.put((b.T if tB else b).copy()), 0.0, hc)
    got = dev.get(hc, (m, n))
    with np.errstate(all="ignore"):
        want = a.astype(np.float64) @ b.astype(np.float64)
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(got[np.isinf(want)], want[np.isinf(want)])
    rows, cols = np.delete(np.arange(m), [7, m - 1])[::50], np.delete(np.arange(n), [3, 1028])[::50]
    check(got, a, b, rows, cols)
