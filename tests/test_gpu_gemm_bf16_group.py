"""The projections of a multi-head attention layer as one call (LINEAR_HEADS_GROUP; csrc/gemm_bf16.hip, gemm_b16_group_kernel):
products of different lengths and sequences in one launch, edges of every tile, what falls back to one after the other."""
import numpy as np
import pytest

from mycaffe_amd.cudadnn import CudaDnnError

pytestmark = pytest.mark.gpu


def round_bf16(a):
    u = np.ascontiguousarray(a, np.float32).view(np.uint32)
    return ((u + 0x7FFF + ((u >> 16) & 1)) & 0xFFFF0000).view(np.float32)


def run(dev, N, K, heads, rows, half, bias=True):
    rng, calls, want = np.random.default_rng(N + K), [], []
    for M, T in rows:
        x, w, b = (rng.standard_normal(s, dtype=np.float32) for s in ((M, K), (N, K), (N,)))
        if half:
            x, w, b = round_bf16(x), round_bf16(w), round_bf16(b)
        y = dev.cuda.AllocMemory(M * N, bHalfSize=half)
        put = lambda a: dev.cuda.AllocMemory(a, bHalfSize=half)  # noqa: E731
        calls.append((M, T, put(x), put(w), put(b) if bias else 0, y))
        r = x.astype(np.float64) @ w.T.astype(np.float64) + (b if bias else 0)
        want.append(r.reshape(M // T, T, heads, N // heads).transpose(0, 2, 1, 3))
    dev.cuda.LinearHeadsGroup(N, K, heads, calls)
    return calls, want


def get(dev, h, n, half):
    if half:
        h, src = dev.zeros(n), h
        dev.cuda.copy(n, src, h)
    return dev.get(h)


# by the estimate, in this order: 256 x 192 tiles, 64 x 64, 128 x 128 with two stages, 64 x 128 with two, the same, 256 x 256, 64 x 64 twice, fp32;
# 128 x 192 on four wavefronts and on eight, 128 x 128 and 64 x 128 with three stages, 128 x 64.  Among them sizes without whole tiles, a
# head size that 16-byte pieces do not divide and too few rows for one launch
@pytest.mark.parametrize("N,K,heads,rows,half", [
    (512, 512, 8, [(4096, 128), (8192, 256), (8192, 256)], True), (256, 256, 4, [(2000, 50), (1000, 40)], True), (768, 768, 12, [(1030, 103), (4100, 100), (3000, 30)], True),
    (512, 512, 8, [(2048, 64), (2048, 64), (2048, 64)], True), (384, 64, 32, [(5000, 100), (77, 7), (1, 1)], True), (1024, 1024, 16, [(8192, 512), (8192, 512)], True),
    (512, 512, 8, [(40, 20), (60, 30)], True), (72, 40, 8, [(130, 13), (65, 5)], True), (96, 96, 6, [(130, 13), (65, 5), (33, 33)], False),
    (1536, 264, 24, [(6000, 100), (2056, 8)], True), (512, 520, 8, [(4104, 27), (4104, 108)], True), (96, 2056, 4, [(8200, 41), (8200, 200)], True),
    (96, 1032, 6, [(8200, 200), (8200, 41)], True), (160, 64, 4, [(4104, 54), (4104, 57)], True)])
def test_projections(dev, N, K, heads, rows, half):
    for bias in (True, False):
        calls, want = run(dev, N, K, heads, rows, half, bias)
        for (M, T, _, _, _, y), w in zip(calls, want):
            got = get(dev, y, M * N, half).reshape(w.shape)
            assert np.abs(got - w).max() <= (2.0 ** -8 if half else 4e-6) * np.abs(w).max()   # one rounding to 16 bits
            if half:
                assert np.sqrt(((got - w) ** 2).mean()) <= 2.0 ** -9 * np.sqrt((w ** 2).mean())


def test_the_same_bits_as_one_by_one(dev):
    N = K = 512
    calls, _ = run(dev, N, K, 8, [(4096, 128), (8192, 256), (8192, 256)], True)
    for M, T, x, w, b, y in calls:
        one = dev.cuda.AllocMemory(M * N, bHalfSize=True)
        dev.cuda.LinearForward(M, N, K, x, w, b, one, T, 8)
        assert np.array_equal(get(dev, one, M * N, True), get(dev, y, M * N, True))


def test_a_result_over_the_next_input(dev):
    # as the calls one after the other: the second product reads what the first one wrote
    M, N = 2048, 256
    rng = np.random.default_rng(0)
    x, w = round_bf16(rng.standard_normal((M, N), dtype=np.float32)), round_bf16(0.05 * rng.standard_normal((N, N), dtype=np.float32))
    hx, hw, hy, hz = (dev.cuda.AllocMemory(a, bHalfSize=True) for a in (x, w, np.zeros(M * N, np.float32), np.zeros(M * N, np.float32)))
    dev.cuda.LinearHeadsGroup(N, N, 1, [(M, M, hx, hw, 0, hy), (M, M, hy, hw, 0, hz)])
    y = round_bf16((x.astype(np.float64) @ w.T.astype(np.float64)).astype(np.float32))
    z = y.astype(np.float64) @ w.T.astype(np.float64)
    assert np.abs(get(dev, hz, M * N, True).reshape(M, N) - z).max() <= 2e-2 * np.abs(z).max()


def test_refused(dev):
    y = dev.zeros(64 * 64)
    p = (64, 8, y, y, 0, y)
    for args in ((64, 64, 7, [p, p]), (64, 64, 8, [p, (64, 9, y, y, 0, y)]), (64, 64, 8, [p]), (64, 64, 8, [p] * 4), (64, 65, 8, [p, p])):
        with pytest.raises(CudaDnnError):
            dev.cuda.LinearHeadsGroup(*args)
