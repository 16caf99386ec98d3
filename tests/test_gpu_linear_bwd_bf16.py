"""Weight and bias gradient of an inner product in one pass, 16-bit storage (csrc/gemm_bf16.hip, b16_tile with SUMS): every tile shape,
contractions cut and not, edges, more stages than turns and fewer; gradients add to what is there."""
import numpy as np
import pytest

from tests.test_gpu_gemm_bf16 import tile

pytestmark = pytest.mark.gpu


def round_bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).view(np.float32)


def get(dev, h, shape):
    f = dev.zeros(int(np.prod(shape)))
    dev.cuda.copy(int(np.prod(shape)), h, f)
    return dev.get(f, shape)


# rows, outputs, inputs
@pytest.mark.parametrize("m,n,k,shape", [
    (1025, 8, 8, 8), (1032, 64, 72, 8), (2000, 96, 200, 8), (8000, 768, 3072, 4), (8000, 3072, 768, 4), (1100, 4096, 1024, 6), (4104, 1000, 264, 8), (1500, 2304, 768, 7),
    (1030, 8192, 4096, 0), (20000, 40, 24, 8), (1088, 50, 64, 8), (1032, 8200, 1032, 1), (1032, 4104, 4104, 2), (1032, 1032, 4104, 3), (4104, 6152, 136, 3),
    (8200, 72, 4104, 5), (2056, 72, 3080, 7), (4104, 136, 3080, 9)])
def test_gradients(dev, m, n, k, shape):
    assert tile(n, k, m)[0] == shape
    rng = np.random.default_rng(m + n)
    x, w, dy, dw, db = (round_bf16(rng.standard_normal(s, dtype=np.float32)) for s in ((m, k), (n, k), (m, n), (n, k), (n,)))
    hx, hw, hdy, hdw, hdb = (dev.cuda.AllocMemory(a, bHalfSize=True) for a in (x, w, dy, dw, db))
    hdx = dev.cuda.AllocMemory(m * k, bHalfSize=True)
    dev.cuda.LinearBackward(m, n, k, hx, hw, hdy, hdw, hdb, hdx)
    got, want = get(dev, hdb, (n,)), db + dy.astype(np.float64).sum(0)
    # one rounding to 16 bits; sums in fp32, at most 128 values and 80 parts one after the other
    assert (np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -24 * (np.abs(db) + 220 * np.sqrt(m))).all()
    want = dw + dy.T @ x   # fp32 sums of products that are exact in it
    assert np.abs(get(dev, hdw, (n, k)) - want).max() <= 2.0 ** -8 * np.abs(want).max()
    want = dy @ w
    assert np.abs(get(dev, hdx, (m, k)) - want).max() <= 2.0 ** -8 * np.abs(want).max()


def test_infinity_reaches_its_sum_alone(dev):
    m, n, k = 4096, 256, 256
    dy = np.ones((m, n), np.float32)
    dy[3000, 17], dy[5, 200] = np.inf, np.nan
    z = np.zeros((m, k), np.float32)
    hx, hw, hdy, hdw, hdb = (dev.cuda.AllocMemory(a, bHalfSize=True) for a in (z, z[:n], dy, z[:n], np.zeros(n, np.float32)))
    dev.cuda.LinearBackward(m, n, k, hx, hw, hdy, hdw, hdb, 0)
    got = get(dev, hdb, (n,))
    assert got[17] == np.inf and np.isnan(got[200]) and (np.delete(got, [17, 200]) == m).all()
