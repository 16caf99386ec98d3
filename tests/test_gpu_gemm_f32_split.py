"""fp32 products on the bf16 matrix cores (csrc/gemm_f32.hip, gemm_f32_split_kernel) where they can go wrong: edges of every tile,
contractions of one or two stages or that end inside one, parts of a contraction, batches and causal operands, values that three bf16
numbers do not hold.  Which tile a size goes to is asked of the library, so that other estimates do not lead a test elsewhere."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

# error of a result over the sum of |a| |b|: the fp32 roundings of at most k / 16 x 6 partial sums (2^-24 each, adding up like a random
# walk, and never more than the running sum), and what the split leaves out (2^-25)
BOUND = lambda k: 2.0 ** -24 * (2 + np.sqrt(6 * k / 16))  # noqa: E731

# from the smallest products taken (2^28 multiplications, 64 k), and the tile that the estimate gives them
SHAPES = [(2052, 4100, 68, 3),      # five stages of one k-step, the last short
          (4100, 3076, 64, 3),      # the shortest contraction, edges in both directions
          (516, 260, 4100, 5),      # parts
          (132, 132, 32004, 5),     # 28 parts of 64 x 64 tiles
          (1000, 4, 140004, 5),     # 32
          (4100, 3076, 292, 0), (3076, 3076, 292, 1), (1028, 4612, 580, 2), (2052, 1544, 612, 3), (2056, 1544, 292, 4), (1028, 1540, 292, 5),
          (1028, 1028, 612, None),  # (32 x 32 tiles, gemm_f32_small_kernel)
          (16004, 388, 100, 3), (580, 7000, 132, 3), (8196, 2308, 76, 3)]


def tile(m, n, k, batch=1, causal=False, heads=False):
    """The number of the tile that the split kernel takes a product with, None where another kernel does."""
    from mycaffe_amd.cudadnn import load_library
    route = load_library().MCH_GemmFloatRoute(m, n, k, batch, 1 * causal + 4 * heads)
    return route // 4 % 16 if route % 4 == 1 else None


def check(got, a, b, rows, cols, alpha=1.0, add=0.0):
    a, b = a[rows].astype(np.float64), b[:, cols].astype(np.float64)
    k = a.shape[1]
    err = np.abs(got[np.ix_(rows, cols)] - alpha * (a @ b) - (add[np.ix_(rows, cols)] if np.ndim(add) else add))
    assert (err / (abs(alpha) * (np.abs(a) @ np.abs(b)) + 1.0)).max() < BOUND(k), (err.max(), k)


def sample(rng, n):
    return np.unique(np.concatenate([[0, 1, n - 1, max(0, n - 4)], rng.integers(0, n, 60)]))


@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k,shape", SHAPES)
def test_edges(dev, m, n, k, shape, tA, tB):
    assert tile(m, n, k) == shape
    rng = np.random.default_rng(m + n + k)
    a, b, c = (rng.standard_normal(s, dtype=np.float32) for s in ((m, k), (k, n), (m, n)))
    ha, hb = dev.put((a.T if tA else a).copy()), dev.put((b.T if tB else b).copy())
    rows, cols = sample(rng, m), sample(rng, n)
    hc = dev.put(c)
    dev.cuda.gemm(tA, tB, m, n, k, -0.5, ha, hb, 1.0, hc)
    check(dev.get(hc, (m, n)), a, b, rows, cols, -0.5, c)
    dev.cuda.gemm(tA, tB, m, n, k, 1.0, ha, hb, 0.0, hc)
    check(dev.get(hc, (m, n)), a, b, rows, cols)


def test_error_is_not_above_that_of_fp32_sums(dev):
    # against 64 bits, relative to a plain fp32 product's error at the same size
    rng = np.random.default_rng(3)
    for m, n, k, shape in ((2048, 4096, 64, 3), (2048, 1024, 288, 5), (2048, 1536, 768, 5), (1024, 1024, 768, None), (512, 256, 8192, 5)):
        assert tile(m, n, k) == shape
        a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((n, k), dtype=np.float32)
        hc = dev.zeros(m * n)
        dev.cuda.gemm(False, True, m, n, k, 1.0, dev.put(a), dev.put(b), 0.0, hc)
        got, rows = dev.get(hc, (m, n)), sample(rng, m)
        want = a[rows].astype(np.float64) @ b.T.astype(np.float64)
        chain = np.zeros((len(rows), n), np.float32)
        for i in range(k):      # one rounding per product
            chain += np.multiply.outer(a[rows, i], b[:, i])
        norm = lambda d: np.sqrt((d ** 2).sum())  # noqa: E731
        assert norm(got[rows] - want) <= 1.02 * norm(chain - want), k


@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False)])
@pytest.mark.parametrize("m,n,k,shape", [(1028, 1540, 612, 5), (2056, 1544, 292, 4), (4100, 3076, 292, 0), (1028, 1028, 612, None)])
def test_values_that_three_parts_do_not_hold(dev, m, n, k, shape, tA, tB):
    assert tile(m, n, k) == shape
    rng = np.random.default_rng(9)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    b[0] = np.where(rng.random(n) < 0.5, 0, 1).astype(np.float32)     # infinities times zero as well
    b[:, 5] = np.abs(b[:, 5])
    big = np.float32(3.4e38)                            # above the largest bf16 number
    a[3, 0], a[200, 7], a[1027, k - 1], a[640, 10] = np.inf, np.nan, -np.inf, big
    a[641, :] = 0
    a[641, 20] = big
    a[700], a[701] = a[700] * np.float32(2.0 ** -120), 0                  # below what the third part holds; zeros
    b[:, 100] *= np.float32(2.0 ** -115)
    ha, hb, hc = dev.put((a.T if tA else a).copy()), dev.put((b.T if tB else b).copy()), dev.zeros(m * n)
    dev.cuda.gemm(tA, tB, m, n, k, 1.0, ha, hb, 0.0, hc)
    got = dev.get(hc, (m, n))
    with np.errstate(all="ignore"):
        a64, b64 = a.astype(np.float64), b.astype(np.float64)
        want = a64 @ b64
        scale = np.abs(a64) @ np.abs(b64)
    assert np.isnan(got[200]).all() and (got[701] == 0).all()
    for r in (3, 1027):
        assert np.array_equal(np.isnan(got[r]), np.isnan(want[r])) and np.array_equal(got[r][~np.isnan(want[r])], want[r][~np.isnan(want[r])])
    fine = np.isfinite(want) & (np.abs(want) < 3e38) & (scale < 3e38)
    fine[[3, 200, 1027]] = False
    assert fine[700].all() and fine[:, 100].sum() >= m - 5 and fine[641].sum() > n / 2
    # 2^-148: results that end among the denormals
    assert (np.abs(got[fine] - want[fine]) <= BOUND(k) * scale[fine] + 2.0 ** -148).all()


# values below 2^-109, of which the parts lose bits or all, times ordinary and very large ones, in either operand
@pytest.mark.parametrize("tA,tB", [(False, True), (False, False), (True, False), (True, True)])
@pytest.mark.parametrize("m,n,k,shape", [(4100, 3076, 292, 0), (3076, 3076, 292, 1), (1028, 4612, 580, 2), (2052, 1540, 612, 3), (2056, 1544, 292, 4),
                                         (2055, 1029, 303, 5), (516, 260, 4100, 5)])
def test_tiny_values_times_large_ones(dev, m, n, k, shape, tA, tB):
    assert tile(m, n, k) == shape
    rng = np.random.default_rng(m + k)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    p2 = lambda e: np.float32(2.0 ** e)  # noqa: E731
    for v, w in ((a.T, b), (b, a.T)):      # columns of the one tiny, of the other large
        v[:, 3] *= p2(-118)
        v[:, 70] *= p2(-125)
        v[:, 130] = (v[:, 130] * p2(-100)) * p2(-34)     # a few bits among the denormals
        v[:, 171] = 0
        v[min(7, k - 1), 171] = p2(-136)
        v[:, 202] = (v[:, 202] * p2(-100)) * p2(-40)     # times 1: a result among the denormals
        w[:, 250], w[:, 251], w[:, 252] = w[:, 250] * p2(60), w[:, 251] * p2(80), w[:, 252] * p2(100)
    ha, hb, hc = dev.put((a.T if tA else a).copy()), dev.put((b.T if tB else b).copy()), dev.zeros(m * n)
    dev.cuda.gemm(tA, tB, m, n, k, 1.0, ha, hb, 0.0, hc)
    got, special = dev.get(hc, (m, n)), [3, 70, 130, 171, 202, 250, 251, 252]
    for rows, cols in ((special, np.arange(n)), (np.arange(m), special), (sample(rng, m), sample(rng, n))):
        at, a64, b64 = np.ix_(rows, cols), a[rows].astype(np.float64), b[:, cols].astype(np.float64)
        want, scale = a64 @ b64, np.abs(a64) @ np.abs(b64)
        fine = scale < 1e38
        assert (np.abs(got[at][fine] - want[fine]) <= BOUND(k) * scale[fine] + k * 2.0 ** -149).all()


# a tiny value in every tile beside ordinary ones: nothing is made over, and nothing has to be
def test_a_stray_tiny_value_changes_nothing(dev):
    m, n, k = 4100, 3076, 292
    assert tile(m, n, k) == 0
    rng = np.random.default_rng(8)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((k, n), dtype=np.float32)
    hb, out = dev.put(b), []
    for tiny in (0.0, 2.0 ** -120, 2.0 ** -140):
        a[::32, 5] = tiny
        hc = dev.zeros(m * n)
        dev.cuda.gemm(False, False, m, n, k, 1.0, dev.put(a), hb, 0.0, hc)
        out.append(dev.get(hc, (m, n)))
    assert np.array_equal(out[0], out[1]) and np.array_equal(out[0], out[2])


@pytest.mark.parametrize("B,T,H,hs,rope", [(3, 700, 12, 64, False), (2, 1024, 12, 64, True), (1, 2044, 6, 48, True)])
def test_into_heads(dev, B, T, H, hs, rope):
    from oracle import attention_ref as R
    C, rng = H * hs, np.random.default_rng(T)
    x, w, b = (rng.standard_normal(s, dtype=np.float32) for s in ((B * T, C), (3 * C, C), (3 * C,)))
    hq = [dev.zeros(B * T * C) for _ in range(3)]
    hr = dev.cuda.CreateRope(0, 0, B * T * C, B, T, H, hs, 10000.0) if rope else 0
    dev.cuda.QkvProjHeads(B, T, H, hs, dev.put(x), dev.put(w), dev.put(b), *hq, hr)
    ref = (x.astype(np.float64) @ w.T.astype(np.float64) + b).reshape(B, T, 3, H, hs)
    for i, h in enumerate(hq):
        want = R.rope_forward(ref[:, :, i], T, H, hs, dtype=np.float64).reshape(B, T, H, hs) if rope and i < 2 else ref[:, :, i]
        # the rotation's angles are fp32
        assert np.abs(dev.get(h, (B, H, T, hs)).transpose(0, 2, 1, 3) - want).max() <= (1e-4 if rope else 4e-6) * np.abs(ref).max()
    if hr:
        dev.cuda.FreeRope(hr)


def test_fp32_sums_on_request(dev):
    # as before there were three parts: whole and head-wise results, and the fused projection
    rng = np.random.default_rng(4)
    B, T, H, hs = 4, 512, 8, 64
    M, K, N = B * T, H * hs, H * hs
    x, w, b = (rng.standard_normal(s, dtype=np.float32) for s in ((M, K), (3 * N, K), (3 * N,)))
    hx, hw, hb = dev.put(x), dev.put(w), dev.put(b)
    want = x.astype(np.float64) @ w.T.astype(np.float64) + b
    out = {}
    for exact in (False, True):
        hy, hq = dev.zeros(M * 3 * N), [dev.zeros(M * N) for _ in range(3)]
        dev.cuda.LinearForward(M, 3 * N, K, hx, hw, hb, hy, bFp32Sums=exact)
        out[exact] = dev.get(hy, (M, 3 * N))
        assert np.abs(out[exact] - want).max() < 4e-6 * np.abs(want).max()
        dev.cuda.QkvProjHeads(B, T, H, hs, hx, hw, hb, *hq, 0, exact)
        heads = [dev.get(h, (B, H, T, hs)).transpose(0, 2, 1, 3).reshape(M, N) for h in hq]
        assert np.array_equal(np.concatenate(heads, 1), out[exact])
        dev.cuda.LinearForward(M, N, K, hx, hw, hb, hy, T, H, exact)
        assert np.abs(dev.get(hy, (M, 3 * N)).ravel()[:M * N].reshape(B, H, T, hs).transpose(0, 2, 1, 3).reshape(M, N) - want[:, :N]).max() < 4e-6 * np.abs(want).max()
    assert not np.array_equal(out[False], out[True])


# the strided products of the attention chain: a batch, and neither operand's nor the result's rows next to each other
# (neither transposed: on the fp32 matrix cores, see k_gemm2)
@pytest.mark.parametrize("tA,tB", [(False, True), (True, False), (True, True), (False, False)])
@pytest.mark.parametrize("outer,m,n,k,shape", [(48, 256, 64, 1020, None), (40, 260, 68, 1000, None), (4, 2052, 1540, 612, 0), (5, 2048, 772, 292, 1), (47, 515, 133, 515, 2), (24, 516, 516, 100, 3), (9, 1027, 1029, 301, 3),
                                               (40, 260, 292, 516, 5)])
def test_batches(dev, outer, m, n, k, shape, tA, tB):
    assert tile(m, n, k, outer) == shape
    rng = np.random.default_rng(outer)
    a, b = rng.standard_normal((outer, m, k), dtype=np.float32), rng.standard_normal((outer, k, n), dtype=np.float32)
    ha, hb = dev.put((a.transpose(0, 2, 1) if tA else a).copy()), dev.put((b.transpose(0, 2, 1) if tB else b).copy())
    hc = dev.zeros(outer * m * n)
    dev.cuda.matmul(outer, m, n, k, ha, hb, hc, 1.0, tA, tB)
    got = dev.get(hc, (outer, m, n))
    for i in (0, outer // 2, outer - 1):
        check(got[i], a[i], b[i], np.arange(m), np.arange(n))


def causal_products(dev, outer, T, hs):
    """P^T dY and V P^T for softmax weights P whose zeros above the diagonal the library knows of, against 64 bits."""
    cuda, rng = dev.cuda, np.random.default_rng(T)
    sc, v = rng.standard_normal((outer, T, T), dtype=np.float32), rng.standard_normal((outer, T, hs), dtype=np.float32)
    hp, hsc, hm = dev.zeros(sc.size), dev.put(sc), dev.put(np.tril(np.ones((T, T), np.float32)))
    hc, d = cuda.CreateCuDNN(), cuda.CreateTensorDesc()
    cuda.SetTensorDesc(d, outer * T, T, 1, 1, False)
    cuda.mask(sc.size, T * T, 0.0, -1e9, hsc, hm, hsc)
    cuda.SoftmaxForward(hc, 1, 0, 1.0, d, hsc, 0.0, d, hp)
    hout = dev.zeros(v.size)
    cuda.matmul(outer, T, hs, T, hp, dev.put(v), hout, 1.0, True, False)
    left = dev.get(hout, v.shape)
    cuda.matmul(outer, hs, T, T, dev.put(v.transpose(0, 2, 1).copy()), hp, hout, 1.0, False, True)
    right = dev.get(hout, (outer, hs, T))
    p = dev.get(hp, sc.shape)
    assert (np.triu(p[0], 1) == 0).all()
    for i in (0, outer // 2, outer - 1):
        check(left[i], p[i].T, v[i], np.arange(T), np.arange(hs))
        check(right[i], v[i].T, p[i].T, np.arange(hs), np.arange(T))


@pytest.mark.parametrize("outer,T,hs,left,right", [(48, 516, 132, 2, 4), (24, 1028, 64, 5, 5), (24, 1027, 67, 3, 3)])
def test_causal_operands(dev, outer, T, hs, left, right):
    assert tile(T, hs, T, outer, causal=True) == left and tile(hs, T, T, outer, causal=True) == right
    causal_products(dev, outer, T, hs)
