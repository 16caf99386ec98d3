"""fp32 products added to a result: its rows are read eight at a time at the end of a tile (csrc/gemm_f32.hip, f32_store)."""
import numpy as np
import pytest

from mycaffe_amd.cudadnn import load_library

pytestmark = pytest.mark.gpu


# edges of the tiles' rows and columns, and the kernel (0 gemm_f32_kernel, 1 gemm_f32_split_kernel, 2 gemm_f32_small_kernel) and tile they go to:
# tile 0 of the split kernel takes one row after the other, as columns do that 16-byte pieces do not divide
SIZES = [(257, 132, 64, 2, 0), (1000, 772, 400, 2, 0), (2049, 516, 300, 2, 0), (130, 4, 900, 2, 0), (65, 8, 700, 2, 0), (1030, 770, 384, 2, 0), (300, 4096, 128, 0, 3), (1100, 2044, 500, 1, 5),
         (301, 2052, 60, 0, 3), (1001, 2052, 40, 0, 1), (4101, 3076, 292, 1, 0), (3077, 3076, 292, 1, 1), (1029, 4612, 580, 1, 2), (2053, 2052, 64, 1, 3), (1001, 3076, 292, 1, 4),
         (1001, 2052, 292, 1, 5), (3077, 3074, 292, 1, 1)]


@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False)])
@pytest.mark.parametrize("m,n,k,kernel,tile", SIZES)
def test_added(dev, m, n, k, kernel, tile, tA, tB):
    c = dev.cuda
    assert load_library().MCH_GemmFloatRoute(m, n, k, 1, 0) == kernel + 4 * tile + 64   # in one part
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
