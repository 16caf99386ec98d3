"""A held-back scaling that goes into a product's alpha (library.hip, Kernel::mem_factor) for factors that are no power of two: either operand,
both, the ends of the range in which it does, the scaled tensor read afterwards."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("fa,fb", [(0.17677669, 1.0), (1.0, 0.3), (0.1, 7.7), (-0.3, 1.0), (3e-8, 1.0), (1e-7, 1.0), (1.5e7, 1.0), (3e7, 1.0), (0.0, 1.0)])
def test_scaling_into_alpha(dev, fa, fb):
    rng = np.random.default_rng(1)
    outer, m, n, k = 3, 65, 130, 97
    a, b = rng.standard_normal((outer, m, k), dtype=np.float32), rng.standard_normal((outer, k, n), dtype=np.float32)
    ha, hb, hc = dev.put(a), dev.put(b), dev.zeros(outer * m * n)
    for h, x, f in ((ha, a, fa), (hb, b, fb)):
        if f != 1.0:
            dev.cuda.scal(x.size, f, h)
    dev.cuda.matmul(outer, m, n, k, ha, hb, hc, 2.0)
    sa, sb = a * np.float32(fa), b * np.float32(fb)
    want, size = 2 * (sa.astype(np.float64) @ sb.astype(np.float64)), 2 * (np.abs(sa.astype(np.float64)) @ np.abs(sb.astype(np.float64)))
    assert (np.abs(dev.get(hc, (outer, m, n)) - want) <= 2.0 ** -24 * (4 + np.sqrt(k)) * size).all()
    assert np.array_equal(dev.get(ha, a.shape), sa) and np.array_equal(dev.get(hb, b.shape), sb)
