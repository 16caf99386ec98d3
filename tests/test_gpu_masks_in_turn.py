"""Masks of several layers that take turns (csrc/library.hip, held_mask_is_causal): what is known of a mask goes with its content, not with
its handle."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_each_softmax_follows_its_own_mask(dev):
    cuda, T, rng = dev.cuda, 96, np.random.default_rng(1)
    hc, d = cuda.CreateCuDNN(), cuda.CreateTensorDesc()
    cuda.SetTensorDesc(d, 2 * T, T, 1, 1, False)
    x, hp = rng.standard_normal((2, T, T), dtype=np.float32), dev.zeros(2 * T * T)
    tril = np.tril(np.ones((T, T), np.float32))
    band = (tril * np.triu(np.ones((T, T), np.float32), -5)).astype(np.float32)
    late = tril.copy()
    late[3, 40] = 1                                     # causal but for one entry
    masks = [tril, band, tril, late, np.ones((T, T), np.float32)]
    handles = [cuda.AllocMemory(m) for m in masks]

    def check(i):
        h = dev.put(x)
        cuda.mask(x.size, T * T, 0.0, -1e29, h, handles[i], h)
        cuda.SoftmaxForward(hc, 1, 0, 1.0, d, h, 0.0, d, hp)
        e = np.where(masks[i] == 0, 0.0, np.exp(x.astype(np.float64)))
        want = e / e.sum(-1, keepdims=True)
        assert np.abs(dev.get(hp, x.shape) - want).max() < 1e-6 and (dev.get(hp, x.shape)[:, masks[i] == 0] == 0).all()

    for i in (0, 1, 2, 3, 4, 0, 3, 1):
        check(i)
    for i, m in ((0, late), (3, tril)):                 # other content behind the same handles
        cuda.SetMemory(handles[i], m)
        masks[i] = m
    for i in (0, 3, 0, 2):
        check(i)
    cuda.FreeMemory(handles[2])                         # and another blob that may get the same handle
    masks[2], handles[2] = band, cuda.AllocMemory(band)
    for i in (2, 0, 2):
        check(i)
    for h in handles:
        cuda.FreeMemory(h)
