"""The gradients of an inner product in one launch, whose tiles are dealt to the XCDs in runs of equal work (csrc/xcd_runs.h): fewer tiles
than XCDs, one product much longer than the other, contractions around the eight stages of a level of sums."""
import numpy as np
import pytest

from mycaffe_amd.cudadnn import load_library
from tests.test_gpu_double import devd  # noqa: F401

pytestmark = pytest.mark.gpu


# rows, outputs, inputs, and how float takes them: 1 one launch, 3 one whose sums are added in levels of eight stages (512 k)
SIZES = [(5, 3, 2, 1), (40, 1536, 384, 3), (256, 1024, 256, 1), (2000, 64, 256, 3), (130, 2304, 768, 3),   # long weight or long data gradient
         (511, 600, 512, 1), (512, 600, 512, 1), (513, 600, 512, 1), (576, 513, 520, 1), (1025, 400, 384, 1), (1029, 401, 387, 1),
         # a level and one more, two whole ones, two and one more, beside contractions below one; in 16-byte pieces and in single values
         (513, 1025, 1536, 3), (1024, 768, 1536, 3), (1025, 513, 1536, 3), (1536, 33, 257, 3), (2049, 64, 256, 3), (33, 2049, 515, 3)]


@pytest.mark.parametrize("base", ["float", "double"])
@pytest.mark.parametrize("m,n,k,route", SIZES)
@pytest.mark.parametrize("accumulate", [False, True])
def test_gradients(dev, devd, base, m, n, k, route, accumulate):  # noqa: F811
    if base == "float":
        assert load_library().MCH_GemmFloatRoute(m, n, k, 1, 16) == route
    t, unit = (np.float32, 2.0 ** -24) if base == "float" else (np.float64, 2.0 ** -53)
    c = dev.cuda if base == "float" else devd.cuda
    rng = np.random.default_rng(m + n + k)
    x, w, dy, dw, db, dx = (rng.standard_normal(s).astype(t) for s in ((m, k), (n, k), (m, n), (n, k), (n,), (m, k)))
    h = [c.AllocMemory(a.ravel()) for a in (x, w, dy, dw, db, dx)]
    c.LinearBackward(m, n, k, *h, accumulate)
    x, w, dy, dw, db, dx = (a.astype(np.float64) for a in (x, w, dy, dw, db, dx))
    # a sum of l products rounds l times at the size of its partial sums, by chance in either direction: sqrt(l) of them in all, and a few at the end
    bound = lambda l: unit * (4 + np.sqrt(l))  # noqa: E731
    for handle, want, scale, l in ((h[3], dw + dy.T @ x, np.abs(dw) + np.abs(dy).T @ np.abs(x), m), (h[4], db + dy.sum(0), np.abs(db) + np.abs(dy).sum(0), m),
                                   (h[5], accumulate * dx + dy @ w, np.abs(dx) + np.abs(dy) @ np.abs(w), n)):
        got = np.asarray(c.GetMemoryFloat(handle, want.size)).reshape(want.shape)
        assert (np.abs(got - want) <= bound(l) * scale).all()
    for a in h:
        c.FreeMemory(a)


@pytest.mark.parametrize("base,m,n,k", [("float", 3667, 280, 188), ("float", 2049, 96, 600), ("float", 2705, 100, 227), ("double", 1367, 77, 160), ("double", 1900, 96, 60),
                                        ("double", 4000, 48, 21)])
def test_error_of_the_bias_gradient(dev, devd, base, m, n, k):  # noqa: F811
    """A bias gradient of many rows is as close to the sum as additions in levels of eight stages leave it."""
    t, unit, quad, lanes = (np.float32, 2.0 ** -24, 4, 8) if base == "float" else (np.float64, 2.0 ** -53, 2, 16)
    c, wide = (dev.cuda, np.float64) if base == "float" else (devd.cuda, np.longdouble)
    if base == "float":
        assert load_library().MCH_GemmFloatRoute(m, n, k, 1, 16) & 1
    rng = np.random.default_rng(m)
    x, w, dy = (rng.standard_normal(s).astype(t) for s in ((m, k), (n, k), (m, n)))
    h = [c.AllocMemory(a.ravel()) for a in (x, w, dy, np.zeros((n, k), t), np.zeros(n, t), np.zeros((m, k), t))]
    c.LinearBackward(m, n, k, *h)
    err = np.asarray(c.GetMemoryFloat(h[4], n)).astype(wide) - dy.astype(wide).sum(0)
    # an addition is off by at most unit / sqrt(3) of its result in the mean square, and sums of N(0, 1) values have their number as mean square:
    # the values of a lane's fragment, 16 of those in a level, its levels, the lanes of a row, the gradient that is added to
    levels = -(-m // 512)
    squares = m / quad * sum(range(2, quad + 1)) + lanes * levels * sum(quad * i for i in range(1, 17)) + lanes * sum(16 * quad * i for i in range(1, levels + 1)) \
        + sum(m / lanes * i for i in range(1, lanes + 1)) + m
    assert np.sqrt((err ** 2).mean()) <= unit * np.sqrt(squares / 3)
    for a in h:
        c.FreeMemory(a)
