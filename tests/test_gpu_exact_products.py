"""What products and convolutions owe without any tolerance, whichever form they take: the sum over nothing; a sum of one term; rows,
columns and images scaled by powers of two; the same results whether or not weights are vouched for."""
import numpy as np
import pytest

from webdnn_amd import hostops as H

pytestmark = pytest.mark.gpu


# (aligned rows, columns in fours: what the planned forms are asked for; odd ones beside them)
@pytest.mark.parametrize("m,n", [(5, 8), (1, 4), (64, 64), (300, 516), (4096, 4096), (7, 6), (5, 9)])
@pytest.mark.parametrize("ta,tb", [(0, 0), (0, 1), (1, 0), (1, 1)])
def test_an_empty_inner_dimension_leaves_the_other_terms(ctx, m, n, ta, tb):
    rng = np.random.default_rng(m + n)
    a, b, c = np.zeros((0, m) if ta else (m, 0), np.float32), np.zeros((n, 0) if tb else (0, n), np.float32), rng.standard_normal(n).astype(np.float32)
    ta_, tb_, tc = (ctx.move_tensor(v) for v in (a, b, c))
    want = np.broadcast_to(np.float32(0.5) * c, (m, n))
    assert (H.gemm(ctx, ta_, tb_, tc, 2.0, 0.5, ta, tb).get_data() == want).all()
    assert (H.gemm(ctx, ta_, tb_, None, 2.0, 0.5, ta, tb).get_data() == 0).all()
    if ta or tb:
        return
    r = rng.standard_normal((m, n)).astype(np.float32)
    assert (H.matmul(ctx, ta_, tb_, tc, ctx.move_tensor(r), "relu").get_data() == np.maximum(c + r, 0)).all()
    x = ctx.move_tensor(np.zeros((3, m, 0), np.float32))   # a batch, which may share its right operand
    assert (H.matmul(ctx, x, tb_, tc).get_data() == c).all()
    assert (H.matmul(ctx, x, ctx.move_tensor(np.zeros((3, 0, n), np.float32))).get_data() == 0).all()


# products and convs with sums of 500 to 4000 terms, enough of them for the forms that large ones take
PRODUCTS = [(2866, 1016, 3336), (3807, 2004, 2736), (4096, 4096, 1024)]
EXPONENTS = [0, -13, -20, -24, -28, -32, -40]


def operands(m, n, k):
    rng = np.random.default_rng(m + n + k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), (rng.standard_normal((k, n)) * 0.03).astype(np.float32)
    a[::7] = np.float32(1.2345678)   # (rows of one value among them, and columns)
    b[:, ::5] = np.float32(0.87654321)
    return rng, a, b


def multiply(ctx, a, b, transposed):
    y = H.gemm(ctx, ctx.move_tensor(a), ctx.move_tensor(np.ascontiguousarray(b.T) if transposed else b), trans_b=int(transposed))
    out = y.get_data()
    y.dispose()
    return out


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("m,n,k", PRODUCTS)
def test_rows_and_columns_of_other_magnitudes_are_the_same_sums(ctx, m, n, k, transposed):
    """A power of two changes no rounding, whatever lies in the rows and columns beside it."""
    rng, a, b = operands(m, n, k)
    want = multiply(ctx, a, b, transposed)
    ea, eb = (2.0 ** rng.choice(EXPONENTS, count).astype(np.float32) for count in (m, n))
    assert (multiply(ctx, a * ea[:, None], b, transposed) == want * ea[:, None]).all()
    assert (multiply(ctx, a, b * eb, transposed) == want * eb).all()


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("m,n,k", PRODUCTS)
def test_a_sum_of_one_term_is_that_product(ctx, m, n, k, transposed):
    rng, a, b = operands(m, n, k)
    few = np.zeros_like(b)
    pick = rng.permutation(max(n, k))[:n] % k
    few[pick, np.arange(n)] = np.float32(0.5)
    assert (multiply(ctx, a, few, transposed) == a[:, pick] * np.float32(0.5)).all()
    few = np.zeros_like(a)
    pick = rng.integers(0, k, m)
    few[np.arange(m), pick] = np.float32(-2)
    assert (multiply(ctx, few, b, transposed) == b[pick] * np.float32(-2)).all()


CONVS = [  # n, c, h, w, cout, kernel, stride
    (32, 1024, 14, 14, 256, 1, 1), (60, 512, 12, 12, 128, 1, 1), (4, 512, 34, 36, 256, 1, 1), (64, 1024, 13, 15, 520, 1, 1), (16, 1024, 28, 28, 512, 1, 2),
    (64, 96, 28, 28, 96, 3, 1), (64, 128, 28, 28, 128, 3, 1), (128, 256, 14, 14, 256, 3, 1), (16, 256, 28, 28, 256, 3, 1), (9, 96, 31, 29, 100, 3, 1)]


def convolve(ctx, x, w, stride, constant=True):
    pads = [w.shape[2] // 2] * 4
    tx, tw = ctx.move_tensor(x), ctx.move_tensor(w)
    y = H.conv(ctx, tx, tw, pads=pads, strides=[stride, stride], constant_weights=constant)
    out = y.get_data()
    for t in (tx, tw, y):
        t.dispose()
    return out


@pytest.mark.parametrize("shape", CONVS)
def test_images_and_channels_of_other_magnitudes_are_the_same_sums(ctx, shape):
    n, c, h, w, cout, kernel, stride = shape
    rng = np.random.default_rng(sum(shape))
    x, wt = rng.standard_normal((n, c, h, w)).astype(np.float32), (rng.standard_normal((cout, c, kernel, kernel)) * 0.03).astype(np.float32)
    x[::3] = np.float32(1.2345678)
    want = convolve(ctx, x, wt, stride)
    ex, ew = (2.0 ** rng.choice(EXPONENTS, (count, 1, 1, 1)).astype(np.float32) for count in (n, cout))
    assert (convolve(ctx, x * ex, wt, stride) == want * ex).all()
    assert (convolve(ctx, x, wt * ew, stride) == want * ew[:, 0]).all()


@pytest.mark.parametrize("shape", CONVS)
def test_weights_that_are_vouched_for_change_no_bits(ctx, shape):
    n, c, h, w, cout, kernel, stride = shape
    rng = np.random.default_rng(sum(shape))
    x, wt = rng.standard_normal((n, c, h, w)).astype(np.float32), (rng.standard_normal((cout, c, kernel, kernel)) * 0.03).astype(np.float32)
    assert (convolve(ctx, x, wt, stride, True) == convolve(ctx, x, wt, stride, False)).all()


@pytest.mark.parametrize("shape", [s for s in CONVS if s[5] == 1 or s[1] < 128])  # (minimal filtering adds inputs before it multiplies them)
def test_a_conv_of_one_tap_moves_channels(ctx, shape):
    n, c, h, w, cout, kernel, stride = shape
    rng = np.random.default_rng(sum(shape))
    x, wt = rng.standard_normal((n, c, h, w)).astype(np.float32), np.zeros((cout, c, kernel, kernel), np.float32)
    pick = rng.integers(0, c, cout)
    wt[np.arange(cout), pick, kernel // 2, kernel // 2] = 1
    assert (convolve(ctx, x, wt, stride) == x[:, pick, ::stride, ::stride]).all()
