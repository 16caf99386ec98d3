"""The gradient of the head layout at more values than one launch numbers (csrc/ew_kernels.hip)."""
import numpy as np
import pytest

from tests.conftest import bf16_round

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,T,H,hs", [(2, 10600000, 5, 13), (3, 7200000, 4, 16)])   # one value a thread, four values a thread
def test_more_values_than_one_launch_numbers(dev, B, T, H, hs):
    C, n = H * hs, B * T * H * hs
    assert 3 * n > 0xf0000000
    period = 1000003
    rng = np.random.default_rng(hs)
    blocks, handles = [], []
    for _ in range(3):
        block = bf16_round(rng.standard_normal(period).astype(np.float32))
        h, src = dev.zeros(n, True), dev.put(block, True)
        dev.cuda.copy(period, src, h)
        have = period
        while have < n:
            more = min(have, n - have)
            dev.cuda.copy(more, h, h, 0, have)
            have += more
        blocks.append(block)
        handles.append(h)
    hx = dev.zeros(3 * n, True)
    dev.cuda.QkvHeadsGrad(B, T, H, hs, *handles, hx)
    rows = B * T
    edge = 0xe0000000 // (3 * C)
    for row in {0, 1, T - 1, T, rows // 2, min(edge - 1, rows - 2), min(edge, rows - 1), rows - 1}:
        v = dev.cuda.CreateMemoryPointer(hx, row * 3 * C, 3 * C)
        got = dev.cuda.GetMemoryFloat(v, 3 * C).reshape(3, H, hs)
        dev.cuda.FreeMemoryPointer(v)
        b, t = divmod(row, T)
        at = ((b * H + np.arange(H)[:, None]) * T + t) * hs + np.arange(hs)[None, :]
        for i in range(3):
            assert np.array_equal(got[i], blocks[i][at % period]), (row, i)
