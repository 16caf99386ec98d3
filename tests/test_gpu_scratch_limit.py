"""Calls where the scratch memory they would like is not to be had: the same results another way."""
import numpy as np
import pytest

from mycaffe_amd.cudadnn import CudaDnn, CudaDnnDouble, CudaDnnError

pytestmark = pytest.mark.gpu


@pytest.fixture(params=[None, 200000])
def limit(request, monkeypatch):
    if request.param:
        monkeypatch.setenv("MYCAFFE_HIP_SCRATCH_LIMIT", str(request.param))
    return request.param


@pytest.mark.parametrize("merged", [False, True])
def test_double_attention_forward(limit, merged):
    cuda, rng = CudaDnnDouble(0), np.random.default_rng(0)
    B, H, T, hs = 2, 3, 130, 16
    q, k, v = (rng.standard_normal((B, H, T, hs)) for _ in range(3))
    hq, hk, hv, hm = (cuda.AllocMemory(a) for a in (q, k, v, np.tril(np.ones((T, T)))))
    hy, hc, ha = cuda.AllocMemory(q.size), cuda.CreateCuDNN(), cuda.CreateAttn()
    cuda.SetAttn(hc, ha, 0, False, B, T, H, hs, 0.0)
    cuda.AttnScaledDotProductForward(hc, ha, T, hq, hk, hv, hm, hy, False, *([T, True] if merged else []))
    s = np.where(np.tril(np.ones((T, T))) == 0, -np.inf, q @ k.transpose(0, 1, 3, 2) / np.sqrt(hs))
    p = np.exp(s - s.max(-1, keepdims=True))
    y = p / p.sum(-1, keepdims=True) @ v
    want = y.transpose(0, 2, 1, 3) if merged else y
    assert np.abs(cuda.GetMemoryFloat(hy).reshape(want.shape) - want).max() <= 1e-13 * np.abs(want).max()
    if limit:   # the gradient has no such form
        with pytest.raises(CudaDnnError):
            cuda.AttnScaledDotProductBackward(hc, ha, hq, hq, hk, hk, hv, hv, hm, hy, hy)
    cuda.Dispose()


@pytest.mark.parametrize("half", [False, True])
def test_products_with_a_long_contraction(limit, half):
    cuda, rng = CudaDnn(0), np.random.default_rng(1)
    M, N, K = 4096, 96, 64

    def put(a):      # through a device copy: host data in 16-bit storage is converted in scratch memory
        h = cuda.AllocMemory(a)
        if half:
            h32, h = h, cuda.AllocMemory(a.size, bHalfSize=True)
            cuda.copy(a.size, h32, h)
        return h

    def get(h, shape):
        h32 = cuda.AllocMemory(int(np.prod(shape)))
        cuda.copy(int(np.prod(shape)), h, h32)
        return cuda.GetMemoryFloat(h32).reshape(shape)

    x, w, dy = (rng.integers(-4, 5, s).astype(np.float32) for s in ((M, K), (N, K), (M, N)))
    hx, hw, hdy = put(x), put(w), put(dy)
    hdw, hdb, hdx, hg, hy = (cuda.AllocMemory(n, bHalfSize=half) for n in (N * K, N, M * K, N * K, M * N))
    cuda.LinearForward(M, N, K, hx, hw, 0, hy)
    cuda.LinearBackward(M, N, K, hx, hw, hdy, hdw, hdb, hdx)
    cuda.gemm(True, False, N, K, M, 1.0, hdy, hx, 0.0, hg)
    # sums of small integers are exact in fp32; 16-bit storage rounds them once
    for h, want in ((hy, x @ w.T), (hdw, dy.T @ x), (hg, dy.T @ x), (hdb, dy.sum(0)), (hdx, dy @ w)):
        assert (np.abs(get(h, want.shape) - want) <= (2.0 ** -8 * np.abs(want) if half else 0)).all()
    cuda.Dispose()
