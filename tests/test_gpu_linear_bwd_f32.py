"""Weight and bias gradient of an inner product in one pass, fp32 (csrc/gemm_f32.hip, gemm_f32_split_kernel with SUMS): every tile shape,
contractions cut and not, edges, more stages than turns and fewer, an odd number of stages; gradients add to what is there."""
import numpy as np
import pytest

from tests.test_gpu_gemm_f32_split import tile

pytestmark = pytest.mark.gpu


# rows, outputs, inputs
@pytest.mark.parametrize("m,n,k,shape", [
    (1032, 640, 640, None), (1000, 512, 1024, None), (700, 1024, 1024, None), (2001, 516, 260, None), (8000, 768, 3072, 0), (8000, 3072, 768, 0), (4100, 2304, 768, 1),
    (1500, 4096, 1024, 3), (20000, 132, 132, 5), (1048, 8192, 4096, 0), (5000, 1024, 64, 5), (70, 4096, 4096, 3), (1028, 1028, 4100, 2), (4100, 136, 4100, 4),
    (4100, 516, 136, 5)])   # None: 32 x 32 tiles
def test_gradients(dev, m, n, k, shape):
    assert tile(n, k, m) == shape
    rng = np.random.default_rng(m + n)
    x, w, dy, dw, db = (rng.standard_normal(s, dtype=np.float32) for s in ((m, k), (n, k), (m, n), (n, k), (n,)))
    hx, hw, hdy, hdw, hdb = (dev.put(a) for a in (x, w, dy, dw, db))
    hdx = dev.zeros(m * k)
    dev.cuda.LinearBackward(m, n, k, hx, hw, hdy, hdw, hdb, hdx)
    got, want = dev.get(hdb, (n,)), db + dy.astype(np.float64).sum(0)
    # at most 128 values in an accumulator, then at most 16 of those and some parts, one after the other
    assert (np.abs(got - want) <= 2.0 ** -24 * (np.abs(want) + 300 * np.sqrt(m))).all()
    rows, cols = rng.integers(0, n, 40), rng.integers(0, k, 40)
    bound = lambda a, b: 2.0 ** -24 * (2 + np.sqrt(a.shape[1])) * (np.abs(a) @ np.abs(b) + 3)  # noqa: E731
    a, b = dy.T[rows].astype(np.float64), x[:, cols].astype(np.float64)
    assert (np.abs(dev.get(hdw, (n, k))[np.ix_(rows, cols)] - dw[np.ix_(rows, cols)] - a @ b) <= bound(a, b)).all()
    rows = rng.integers(0, m, 40)
    a, b = dy[rows].astype(np.float64), w[:, cols].astype(np.float64)
    assert (np.abs(dev.get(hdx, (m, k))[np.ix_(rows, cols)] - a @ b) <= bound(a, b)).all()


def test_infinity_reaches_its_sum_alone(dev):
    m, n, k = 4096, 512, 512
    dy = np.ones((m, n), np.float32)
    dy[3000, 17], dy[5, 200] = np.inf, np.nan
    z = np.zeros((m, k), np.float32)
    hx, hw, hdy, hdw, hdb = (dev.put(a) for a in (z, z[:n], dy, z[:n], np.zeros(n, np.float32)))
    dev.cuda.LinearBackward(m, n, k, hx, hw, hdy, hdw, hdb, 0)
    got = dev.get(hdb, (n,))
    assert got[17] == np.inf and np.isnan(got[200]) and (np.delete(got, [17, 200]) == m).all()
