"""16-bit products whose tiles keep three and four stages in LDS (csrc/gemm_bf16.hip, b16_tile with S > 2): contractions shorter than the
stages, that end inside one, one stage more than the ring; sizes with edges for each of these tiles; all layouts."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def round_bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).view(np.float32)


# 64 x 64 and 128 x 64 tiles; 64 x 128 with two and three stages; 128 x 128 with three; 128 x 192 on eight wavefronts; parts
@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False)])
@pytest.mark.parametrize("m,n", [(72, 72), (520, 264), (480, 2056), (2056, 1544), (1000, 776), (1304, 2056), (3208, 776), (8008, 520), (4104, 1288)])
def test_contractions(dev, m, n, tA, tB):
    for k in (8, 64, 72, 128, 136, 192, 200, 256, 264, 520, 1032, 2056):
        if m * n > 4e6 and k > 600:
            continue
        rng = np.random.default_rng(m + n + k)
        a, b, c = (round_bf16(rng.standard_normal(s, dtype=np.float32)) for s in ((m, k), (k, n), (m, n)))
        put = lambda x: dev.cuda.AllocMemory(np.ascontiguousarray(x), bHalfSize=True)  # noqa: E731
        ha, hb, hc, hf = put(a.T if tA else a), put(b.T if tB else b), put(c), dev.zeros(m * n)
        dev.cuda.gemm(tA, tB, m, n, k, 0.5, ha, hb, 1.0, hc)
        dev.cuda.copy(m * n, hc, hf)
        got = dev.get(hf, (m, n))
        want, size = 0.5 * (a @ b) + c, 0.5 * (np.abs(a) @ np.abs(b)) + np.abs(c)
        # one rounding to 16 bits; fp32 sums on both sides
        assert (np.abs(got - want) <= 2.0 ** -8 * np.abs(want) + 2.0 ** -22 * np.sqrt(k) * size + 1e-30).all(), k
        for h in (ha, hb, hc, hf):
            dev.cuda.FreeMemory(h)
