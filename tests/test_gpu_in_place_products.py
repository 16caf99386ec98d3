"""Products whose result lies in the memory of an operand, at sizes where that is right: one workgroup reads all that it overwrites (one
tile; the rows of A in place, one tile wide; the columns of B in place, one tile high), or the contraction is cut into parts.  The
kernels of smaller tiles have several workgroups there and must not take them."""
import numpy as np
import pytest

from tests.test_gpu_block_fused import side  # noqa: F401  (the three storage types)

pytestmark = pytest.mark.gpu

# (m, n, k), and the operand that the result lies in.  Tiles of floats are 64 wide and high at least, of doubles 32.
SIZES = {
    "float": [(32, 64, 64, "A"), (17, 64, 64, "B"), (64, 64, 64, "A"), (64, 64, 64, "B"), (33, 40, 40, "A"), (64, 64, 512, "A"), (40, 48, 2048, "A"),
              (48, 40, 2048, "B"), (2000, 64, 64, "A"), (2000, 40, 40, "A"), (64, 2000, 64, "B"), (100, 2048, 2048, "A"), (2048, 100, 2048, "B")],
    "bf16": [(40, 64, 64, "A"), (16, 64, 64, "B"), (64, 64, 64, "A"), (64, 64, 64, "B"), (128, 128, 128, "A"), (2000, 128, 128, "A"), (128, 2000, 128, "B"),
             (120, 1408, 1408, "A"), (1408, 120, 1408, "B"), (8, 5632, 1408, "B"), (40, 5248, 1408, "B")],
    "double": [(32, 32, 32, "A"), (32, 32, 32, "B"), (17, 32, 32, "B"), (30, 30, 30, "A"), (2000, 32, 32, "A"), (32, 2000, 32, "B"), (20, 32, 256, "A")],
}


def check(s, h, want, scale, k):
    got = s.cuda.GetMemoryFloat(h, want.size) if s.kind == "double" else s.dev.get(h)[:want.size]
    unit = 2.0 ** -53 if s.kind == "double" else 2.0 ** -24
    # the sums' roundings, and one to 16 bits
    assert (np.abs(got.reshape(want.shape) - want) <= unit * (4 + np.sqrt(k)) * scale + (2.0 ** -8 * np.abs(want) if s.half else 0)).all()


@pytest.mark.parametrize("at", range(max(len(v) for v in SIZES.values())))
def test_product_over_an_operand(side, at):  # noqa: F811
    if at >= len(SIZES[side.kind]):
        pytest.skip("no such size")
    m, n, k, over = SIZES[side.kind][at]
    rng = np.random.default_rng(m + n + k)
    tB = over == "B" and m != k   # stored (n, k); the columns of B in place where it is stored (k, n)
    (ha, a), (hb, b) = side.put(rng.standard_normal((m, k))), side.put(rng.standard_normal((n, k) if tB else (k, n)))
    b = b.T if tB else b
    hc = ha if over == "A" else hb
    side.cuda.gemm(False, tB, m, n, k, 1.0, ha, hb, 0.0, hc)
    check(side, hc, a @ b, np.abs(a) @ np.abs(b), k)


@pytest.mark.parametrize("kind", ["whole", "heads", "projections", "gradient", "weight gradient"])
def test_calls_of_an_inner_product_over_an_operand(side, kind):  # noqa: F811
    rng = np.random.default_rng(5)
    n = 32 if side.kind == "double" else 64
    (hx, x), (hw, w), (hb, b), (hdy, dy) = (side.put(rng.standard_normal(s)) for s in ((n, n), (n, n), (n,), (n, n)))
    want, scale = x @ w.T + b, np.abs(x) @ np.abs(w.T) + np.abs(b)
    if kind == "whole":
        side.cuda.LinearForward(n, n, n, hx, hw, hb, hx)
        check(side, hx, want, scale, n)
    elif kind == "heads":
        heads = lambda v: v.reshape(2, n // 2, 4, n // 4).transpose(0, 2, 1, 3)  # noqa: E731
        side.cuda.LinearForward(n, n, n, hx, hw, hb, hx, n // 2, 4)
        check(side, hx, heads(want), heads(scale), n)
    elif kind == "projections":   # n / 4 wide: the product is one tile
        C = n // 4
        (hx, x), (hw, w), (hb, b) = (side.put(rng.standard_normal(s)) for s in ((n, C), (3 * C, C), (3 * C,)))
        hk, hv = side.zeros(n * C), side.zeros(n * C)
        side.cuda.QkvProjHeads(2, n // 2, 2, C // 2, hx, hw, hb, hx, hk, hv)
        for i, h in enumerate((hx, hk, hv)):
            part = slice(i * C, (i + 1) * C)
            heads = lambda v: v[:, part].reshape(2, n // 2, 2, C // 2).transpose(0, 2, 1, 3)  # noqa: E731
            check(side, h, heads(x @ w.T + b), heads(np.abs(x) @ np.abs(w.T) + np.abs(b)), C)
    elif kind == "gradient":
        hdw, hdb = side.zeros(n * n), side.zeros(n)
        side.cuda.LinearBackward(n, n, n, hx, hw, hdy, hdw, hdb, hdy)
        check(side, hdy, dy @ w, np.abs(dy) @ np.abs(w), n)
        check(side, hdw, dy.T @ x, np.abs(dy.T) @ np.abs(x), n)
        check(side, hdb, dy.sum(0), np.abs(dy).sum(0), n)
    else:                         # the weight gradient over the input, which it is added to
        side.cuda.LinearBackward(n, n, n, hx, hw, hdy, hx, 0, 0)
        check(side, hx, x + dy.T @ x, np.abs(x) + np.abs(dy.T) @ np.abs(x), n)


# matrices of a batch, each over its own operand
@pytest.mark.parametrize("over", ["A", "B"])
def test_batch_over_an_operand(side, over):  # noqa: F811
    if side.half:
        pytest.skip("strided products are of floats and doubles")
    n = 32 if side.kind == "double" else 64
    rng = np.random.default_rng(6)
    (ha, a), (hb, b) = (side.put(rng.standard_normal((5, n, n))) for _ in range(2))
    hc = ha if over == "A" else hb
    side.cuda.matmul(5, n, n, n, ha, hb, hc)
    check(side, hc, a @ b, np.abs(a) @ np.abs(b), n)
