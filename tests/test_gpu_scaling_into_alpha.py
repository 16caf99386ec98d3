"""A held-back scaling of a product's operand (library.hip, Kernel::mem_factor), whether it goes into alpha or is applied first: either operand,
both, factors of every size, the scaled tensor read afterwards, values near the end of the range."""
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


# the unscaled sums are past the largest fp32 number, the scaled operand's are not: factors that are no power of two, and those that are
# too far from 1
@pytest.mark.parametrize("size,f,other", [(1e35, 1e-6, 1e4), (1e35, 2.0 ** -20, 1e4), (1e38, 0.17677669, 1.0), (1.2e38, 0.3, 1.0), (1e-42, 1e6, 1.0)])
@pytest.mark.parametrize("first", [True, False])
def test_scaled_operands_near_the_end_of_the_range(dev, size, f, other, first):
    rng = np.random.default_rng(2)
    outer, m, k = 2, 48, 64 if size < 1e38 else 5
    a, b = (rng.uniform(0.5, 1, (outer, m, k)) * size / k * 8).astype(np.float32), (rng.uniform(0.5, 1, (outer, k, m)) * other).astype(np.float32)
    ha, hb, hc = dev.put(a), dev.put(b), dev.zeros(outer * m * m)
    dev.cuda.scal(a.size, f, ha)
    if first:
        dev.cuda.matmul(outer, m, m, k, ha, hb, hc)
    else:   # the scaled tensor as the second operand
        a, b = a.reshape(outer, k, m), b.reshape(outer, m, k)
        dev.cuda.matmul(outer, m, m, k, hb, ha, hc)
        a, b = b, a
    scaled = a.astype(np.float64) @ b.astype(np.float64) * np.float32(f)
    assert np.abs(scaled).max() < 3.4e38
    got = dev.get(hc, scaled.shape)
    # one rounding of every scaled value besides the sums'
    assert (np.abs(got - scaled) <= 2.0 ** -24 * (5 + np.sqrt(k)) * np.abs(scaled)).all()
