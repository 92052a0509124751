"""Products cut along K whose chunk sums a second kernel adds, against sums in 64 bits."""
import numpy as np
import pytest

from webdnn_amd import capi
from webdnn_amd import hostops as H

pytestmark = pytest.mark.gpu


def within(got, a, b, extra):
    """A chain of at most k roundings of half an ulp of the sum of magnitudes, and three more for the epilogue."""
    a, b = a.astype(np.float64), b.astype(np.float64)
    want = a @ b + extra
    bound = (a.shape[-1] + 4) * 2.0 ** -24 * (np.abs(a) @ np.abs(b) + np.abs(extra))
    return (np.abs(got - np.maximum(want, 0.0)) <= bound).all()


# around the line between one workgroup a block and cut tiles, whole and ragged
@pytest.mark.parametrize("m,n,k", [(384, 768, 3072), (257, 1025, 2560), (288, 928, 2559), (500, 514, 4099), (256, 1024, 2560), (33, 4127, 5000)])
def test_long_k_with_residual(ctx, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    bias, r = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    ta, tb, tbias, tr = (ctx.move_tensor(v) for v in (a, b, bias, r))
    got = H.matmul(ctx, ta, tb, tbias, tr, "relu").get_data()
    assert within(got, a, b, bias.astype(np.float64) + r)
    got = H.gemm(ctx, ta, ctx.move_tensor(np.ascontiguousarray(b.T)), tbias, 1.0, 1.0, 0, 1, epilogue="relu").get_data()
    assert within(got, a, b, bias.astype(np.float64))


# which form serves on either side of each line, B n-contiguous and k-contiguous
@pytest.mark.parametrize("m,n,k,plain,transposed", [(384, 768, 3072, True, True), (384, 768, 2816, True, True), (384, 768, 2815, True, True),
                                                   (384, 768, 2812, False, True), (384, 1024, 2047, True, True), (384, 1024, 2000, False, False),
                                                   (500, 1024, 2048, False, False), (500, 1024, 2560, False, True), (500, 1024, 4096, True, True),
                                                   (500, 1024, 4092, False, True), (530, 1024, 2304, True, True), (530, 1024, 2300, False, True),
                                                   (530, 1024, 2044, False, False), (700, 1024, 1023, False, True), (1000, 768, 3072, True, True),
                                                   (1000, 768, 3068, False, True), (1000, 1024, 4096, False, True), (256, 1024, 4096, False, False)])
def test_which_form_long_products_take(ctx, m, n, k, plain, transposed):
    a, b = ctx.empty_tensor([m, k]), ctx.empty_tensor([n, k])
    H.gemm(ctx, a, b.alias([k, n])).dispose()
    assert (ctx.last_plan()["tile"] == "64x64") == plain, ctx.last_plan()
    H.gemm(ctx, a, b, trans_b=1).dispose()
    assert (ctx.last_plan()["tile"] == "64x64") == transposed, ctx.last_plan()


@pytest.mark.parametrize("m,n,k", [(384, 768, 3072), (530, 1024, 2304), (700, 1024, 4100)])
@pytest.mark.parametrize("transposed", [0, 1])
def test_cut_tiles_round_no_more_than_sixteen_chains(ctx, m, n, k, transposed):
    """A result is the sum of sixteen chains of one rounding a product, as in the one-launch form that the tiles stand in for."""
    rng = np.random.default_rng(m + k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    got = H.gemm(ctx, ctx.move_tensor(a), ctx.move_tensor(np.ascontiguousarray(b.T) if transposed else b), trans_b=transposed).get_data()
    assert ctx.last_plan()["tile"] == "64x64" and ctx.last_plan()["split"] == 16, ctx.last_plan()
    a64, b64 = a[:64].astype(np.float64), b[:, :128].astype(np.float64)
    chunk = -(-(-(-k // 16)) // 16) * 16
    want, chains = a64 @ b64, np.zeros((64, 128), np.float32)
    for first in range(0, k, chunk):
        acc = np.zeros((64, 128), np.float32)
        for i in range(first, min(first + chunk, k)):
            acc = (acc + np.outer(a64[:, i], b64[i])).astype(np.float32)
        chains += acc
    # the same roundings in another order: over 8192 results the two norms differ by a few per cent
    assert np.linalg.norm(got[:64, :128] - want) <= 1.1 * np.linalg.norm(chains - want)


def test_no_room_for_the_chunk_sums(ctx):
    """Without memory for the workspace of cut tiles the product runs in one launch, and no error stays behind."""
    rng = np.random.default_rng(3)
    a, b = rng.standard_normal((384, 3072)).astype(np.float32), rng.standard_normal((3072, 768)).astype(np.float32)
    ta, tb, mine = ctx.move_tensor(a), ctx.move_tensor(b), ctx.empty_tensor([384, 768])
    H.matmul(ctx, ta, tb).dispose()
    assert ctx.last_plan()["split"] > 1 and ctx.last_plan()["tile"] == "64x64"
    ctx.sync()
    capi.call("wdh_trim", 0)
    ctx.set_option("memory_limit_mib", 1)
    try:
        mine.dispose()  # (the one block the pool has: the result takes it, and no other fits)
        y = H.matmul(ctx, ta, tb, epilogue="relu")
        assert ctx.last_plan()["tile"] == "32x32" and capi.last_error() == ""
    finally:
        ctx.set_option("memory_limit_mib", 0)
    assert within(y.get_data(), a, b, np.zeros(768))


# chunk counts below, at and above the eight requested at a time and twice that, two slabs of 16 channels a chunk; planes
# whose quads are whole and ragged; groups
@pytest.mark.parametrize("split", [2, 7, 8, 9, 16, 17])
@pytest.mark.parametrize("cout,h,w,group", [(24, 8, 8, 1), (70, 7, 7, 1), (12, 6, 10, 2), (5, 1, 3, 1)])
def test_cut_conv_with_residual(ctx, split, cout, h, w, group):
    c = 32 * split * group
    rng = np.random.default_rng(split * 1000 + c + h)
    x = rng.standard_normal((3, c, h, w)).astype(np.float32)
    wt, bias = rng.standard_normal((cout, c // group, 1, 1)).astype(np.float32), rng.standard_normal(cout).astype(np.float32)
    r = rng.standard_normal((3, cout, h, w)).astype(np.float32)
    ctx.set_option("split_k", split)
    try:
        got = H.conv(ctx, ctx.move_tensor(x), ctx.move_tensor(wt), ctx.move_tensor(bias), None, group, None, [0] * 4, [1, 1],
                     epilogue="relu", residual=ctx.move_tensor(r)).get_data()
        plan = ctx.last_plan()
    finally:
        ctx.set_option("split_k", -1)
    assert plan["split"] == split and plan["split_tiles"] > 0, plan
    cg, og = c // group, cout // group
    for i in range(3):
        for g in range(group):
            o = slice(g * og, (g + 1) * og)
            extra = bias[o, None].astype(np.float64) + r[i, o].reshape(og, -1)
            assert within(got[i, o].reshape(og, -1), wt[o, :, 0, 0], x[i, g * cg:(g + 1) * cg].reshape(cg, -1), extra)
