"""GEMM operands of 2 GiB and more: the tile kernels address a tile or a stage with 32-bit offsets from its own beginning, so
an operand's size does not change the kernel (csrc/gemm_f32.hip, gemm_bf16.hip)."""
import numpy as np
import pytest

from tests.conftest import bf16_round

pytestmark = pytest.mark.gpu

PERIOD = 1000   # rows of the repeated block; no power of two, so that an address that wraps at 2 or 4 GiB hits other rows


def big_operand(dev, rows, cols, half, rng):
    block = bf16_round(rng.standard_normal((PERIOD, cols)).astype(np.float32))
    h, src, n = dev.zeros(rows * cols, half), dev.put(block, half), rows * cols
    dev.cuda.copy(block.size, src, h)
    have = block.size
    while have < n:
        more = min(have, n - have)
        dev.cuda.copy(more, h, h, 0, have)
        have += more
    return h, block


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("side", ["A", "B"])
def test_many_rows_of_a_short_contraction(dev, side, half):
    k, small, limit = 256, 8, (1 << 22 if half else 1 << 21)
    rows = limit + 40
    rng = np.random.default_rng(1)
    h, block = big_operand(dev, rows, k, half, rng)
    s = bf16_round(rng.standard_normal((small, k)).astype(np.float32))
    hs, hc = dev.put(s, half), dev.zeros(rows * small, half)
    args = (rows, small, k) if side == "A" else (small, rows, k)
    dev.cuda.gemm(False, True, *args, 1.0, *((h, hs) if side == "A" else (hs, h)), 0.0, hc)
    got = dev.get(hc, args[:2])
    got = got if side == "A" else got.T
    ref = np.resize(block.astype(np.float64) @ s.T.astype(np.float64), (rows, small))
    assert np.abs(got - ref).max() <= (2.0 ** -8 if half else 2e-6) * np.abs(ref).max()
    # the same kernel as for an operand just below 2 GiB: the time goes with the rows
    from mycaffe_amd.cudadnn import CUDAFN
    ms = [min(dev.cuda.TimeFunction(CUDAFN.CUDA_GEMM, [1.0, 0.0], [0, 1] + ([r, small] if side == "A" else [small, r]) + [k, 0] +
                                    ([h, hs] if side == "A" else [hs, h]) + [0, hc], 2, 3) for _ in range(3)) for r in (limit - 100, rows)]
    assert ms[1] < 2.0 * ms[0], ms


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("side", ["A", "B"])
def test_wide_rows_of_a_long_contraction(dev, side, half):
    """The operand lies with its row index at unit stride: a weight gradient of a large vocabulary."""
    wide, small, k = 16640, 8, (65544 if half else 32776)
    rng = np.random.default_rng(2)
    h, block = big_operand(dev, k, wide, half, rng)
    s = bf16_round(rng.standard_normal((k, small)).astype(np.float32))
    hs, hc = dev.put(s, half), dev.zeros(wide * small, half)
    args = (wide, small, k) if side == "A" else (small, wide, k)
    dev.cuda.gemm(True, False, *args, 1.0, *((h, hs) if side == "A" else (hs, h)), 0.0, hc)
    got = dev.get(hc, args[:2])
    got = got if side == "A" else got.T
    pad = np.zeros((-(-k // PERIOD) * PERIOD, small))
    pad[:k] = s
    ref = block.T.astype(np.float64) @ pad.reshape(-1, PERIOD, small).sum(0)
    assert np.abs(got - ref).max() <= (2.0 ** -8 if half else 3e-5) * np.abs(ref).max()
