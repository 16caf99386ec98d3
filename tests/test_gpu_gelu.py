"""The tanh form of GELU through the logistic function's smaller tail (csrc/ew_kernels.hip, GeluF and GeluGradF): both signs, the tails,
what infinities and NaN give, sizes around the eight elements of a trip."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 7, 8, 9, 4099, 1 << 21])
def test_against_float64(dev, n):
    x = np.linspace(-9, 9, n).astype(np.float32) if n > 9 else np.linspace(-2, 3, n).astype(np.float32)
    hx, hy, hg, hdx = dev.put(x), dev.zeros(n), dev.put(np.ones(n, np.float32)), dev.zeros(n)
    dev.cuda.gelu_fwd(n, hx, hy, True)
    dev.cuda.gelu_bwd(n, hg, hy, hdx, hx, True)
    x = x.astype(np.float64)
    u, ug = np.sqrt(2 / np.pi) * (x + 0.044715 * x ** 3), 0.797885 * (x + 0.044715 * x ** 3)
    want, s = x / (1 + np.exp(-2 * u)), 1 / (1 + np.exp(-2 * ug))
    # the exponent 2 u is off by four roundings of itself (the constants, the square, the sum, the product), the rest by a few units in the
    # last place
    eps = 2.0 ** -24
    assert (np.abs(dev.get(hy) - want) <= (4 + 8 * np.abs(u)) * eps * np.abs(want) + 1e-37).all()
    poly = np.abs(0.0535161 * x ** 3 + 0.398942 * x) * 4 * s * (1 - s)
    want = s + (0.0535161 * x ** 3 + 0.398942 * x) * 4 * s * (1 - s)
    assert (np.abs(dev.get(hdx) - want) <= (8 + 8 * np.abs(ug)) * eps * (s + poly)).all()


def test_infinities_and_nan(dev):
    x = np.array([np.inf, -np.inf, np.nan, 0.0, -0.0, 300.0, -300.0, 3e38], np.float32)
    hx, hy = dev.put(x), dev.zeros(8)
    dev.cuda.gelu_fwd(8, hx, hy, True)
    y = dev.get(hy)
    assert y[0] == np.inf and np.isnan(y[1]) and np.isnan(y[2]) and y[3] == 0 and y[4] == 0 and y[5] == 300 and y[6] == 0 and y[7] == x[7]
