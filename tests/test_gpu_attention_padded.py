"""Attention of head sizes that the matrix-core kernels pad (csrc/attn_prefill.hip, csrc/attn_backward.hip with PADDED): sizes around each
kernel's, every kind of mask, lengths around the tiles, what lies past a row."""
import numpy as np
import pytest

from oracle import attention_ref as R
from tests.conftest import BF16_RTOL, FP32_RTOL, bf16_round
from tests.test_gpu_attention_backward import _check, _fwd_bwd

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [False, True])
@pytest.mark.parametrize("hs", [4, 8, 16, 24, 32, 40, 48, 56, 72, 96, 120])
@pytest.mark.parametrize("B,H,Tq,Tk", [(2, 3, 130, 130), (1, 2, 65, 200), (1, 1, 1, 1), (3, 2, 31, 33)])
def test_masks(dev, B, H, Tq, Tk, hs, half):
    rng = np.random.default_rng(hs + Tq)
    q, dy = (bf16_round(rng.standard_normal((B, H, Tq, hs)).astype(np.float32)) for _ in range(2))
    k, v = (bf16_round(rng.standard_normal((B, H, Tk, hs)).astype(np.float32)) for _ in range(2))
    tol = BF16_RTOL if half else FP32_RTOL
    keys = (rng.random((B, Tk)) < 0.7).astype(np.float32)
    keys[0, 0] = 1
    if B > 2:
        keys[2] = 0      # masked everywhere: uniform weights
    batch = (rng.random((B, Tq, Tk)) < 0.6).astype(np.float32)
    batch[:, :, 0] = 1
    for mask, kind in ([(R.causal_mask(Tq), 0)] if Tq == Tk else []) + [(None, 0), (keys, 1), (batch, 2)]:
        _check(_fwd_bwd(dev, q, k, v, dy, mask, kind, half), q, k, v, dy, mask, kind, tol, "kind %d" % kind)


def test_infinite_neighbours(dev):
    # a row is padded with zeros, not with what lies behind it: -inf in a key keeps its weight at zero, and its row's neighbours unharmed
    rng = np.random.default_rng(3)
    q, k, v = (np.abs(rng.standard_normal((1, 1, 64, 16))).astype(np.float32) for _ in range(3))
    k[0, 0, 20, 3] = -np.inf
    hc, ha = dev.cuda.CreateCuDNN(), dev.cuda.CreateAttn()
    dev.cuda.SetAttn(hc, ha, 0, False, 1, 64, 1, 16, 0.0)
    hy = dev.zeros(q.size)
    dev.cuda.AttnScaledDotProductForward(hc, ha, 64, dev.put(q), dev.put(k), dev.put(v), 0, hy, 0)
    keep = np.delete(np.arange(64), 20)
    want = R.softmax_lastaxis(q.astype(np.float64) @ k[:, :, keep].swapaxes(-1, -2) / 4, np.float64) @ v[:, :, keep]
    assert np.abs(dev.get(hy, q.shape) - want).max() <= 1e-5 * np.abs(want).max()
    dev.cuda.FreeAttn(ha)
    dev.cuda.FreeCuDNN(hc)
