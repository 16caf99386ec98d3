"""fp32 products added to a result: its rows are read eight at a time at the end of a tile (csrc/gemm_f32.hip, f32_store)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# edges of the tiles' rows and columns; columns that 16-byte pieces do not divide (one row after the other); rows 16 KB apart
@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False)])
@pytest.mark.parametrize("m,n,k", [(257, 132, 64), (1000, 772, 400), (2049, 516, 300), (130, 4, 900), (65, 8, 700), (1030, 770, 384), (300, 4096, 128), (1100, 2044, 500)])
def test_added(dev, m, n, k, tA, tB):
    c = dev.cuda
    rng = np.random.default_rng(m + n + k)
    a, b, old = (rng.standard_normal(s).astype(np.float32) for s in ((m, k), (k, n), (m, n)))
    h = [c.AllocMemory(np.ascontiguousarray(x).ravel()) for x in (a.T if tA else a, b.T if tB else b, old)]
    c.gemm(tA, tB, m, n, k, 0.5, h[0], h[1], -2.0, h[2])
    got = np.asarray(c.GetMemoryFloat(h[2], m * n)).reshape(m, n)
    want = 0.5 * (a.astype(np.float64) @ b) - 2.0 * old
    # sqrt(k) roundings of the products' size by chance, and those of the scaling and the sum
    bound = 2.0 ** -24 * (4 + np.sqrt(k)) * (np.abs(a).astype(np.float64) @ np.abs(b) + 2 * np.abs(old))
    assert (np.abs(got - want) <= bound).all()
    for x in h:
        c.FreeMemory(x)
