"""Products on the bf16 matrix cores (operands split into three bfloat16 parts) against sums in 64 bits and against the fp32
instruction."""
import numpy as np
import pytest

from webdnn_amd import capi
from webdnn_amd import hostops as H

pytestmark = pytest.mark.gpu

TILES = {3: "128x128", 4: "64x128", 5: "128x64", 6: "64x64", 7: "256x128", 8: "64x64", 9: "64x64"}


@pytest.fixture
def split(ctx):
    yield lambda value: ctx.set_option("split_products", value)
    for name, value in (("split_products", 1), ("split_k", -1), ("conv3x3_winograd", 1), ("conv1x1_stride2_in_place", 1)):
        ctx.set_option(name, value)


def product(ctx, a, b, transposed, bias=None, r=None, epilogue=None):
    tb = ctx.move_tensor(np.ascontiguousarray(b.T) if transposed else b)
    if r is not None:
        return H.matmul(ctx, ctx.move_tensor(a), tb, ctx.move_tensor(bias), ctx.move_tensor(r), epilogue).get_data()
    return H.gemm(ctx, ctx.move_tensor(a), tb, None if bias is None else ctx.move_tensor(bias), trans_b=int(transposed), epilogue=epilogue).get_data()


def within(got, want, magnitudes, k):
    """A chain of at most k roundings of half an ulp of the sum of magnitudes, and a few more for the two sums and the epilogue."""
    return (np.abs(got - want) <= (k + 8) * 2.0 ** -24 * magnitudes + 1e-37).all()


# one slab, a ragged last one, two to five slabs (the loop's prologue and tail), edges of every tile in both directions
@pytest.mark.parametrize("mode", sorted(TILES))
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("m,n,k", [(64, 64, 16), (1, 4, 20), (65, 132, 32), (128, 128, 48), (129, 68, 64), (257, 260, 76), (256, 256, 80), (63, 516, 644)])
def test_tiles_and_edges(ctx, split, mode, transposed, m, n, k):
    rng = np.random.default_rng(m + n + k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, n)).astype(np.float32)
    bias, r = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    split(mode)
    ctx.set_option("gemm_wavesplit", 0)  # (and one row goes to the kernel of few rows otherwise)
    try:
        got = product(ctx, a, b, transposed, bias, None if transposed else r, "relu")
    finally:
        ctx.set_option("gemm_wavesplit", 1)
    assert ctx.last_plan()["tile"] == TILES[mode], ctx.last_plan()
    a, b = a.astype(np.float64), b.astype(np.float64)
    extra = bias + (0.0 if transposed else r)
    assert within(got, np.maximum(a @ b + extra, 0), np.abs(a) @ np.abs(b) + np.abs(extra), k)


@pytest.mark.parametrize("mode", sorted(TILES))
@pytest.mark.parametrize("chunks", [2, 5, 16])
def test_cut_along_k(ctx, split, mode, chunks):
    rng = np.random.default_rng(chunks)
    a, b = rng.standard_normal((150, 1044)).astype(np.float32), rng.standard_normal((1044, 200)).astype(np.float32)
    split(mode)
    ctx.set_option("split_k", chunks)
    got = product(ctx, a, b, False)
    assert ctx.last_plan()["tile"] == TILES[mode] and ctx.last_plan()["split"] > 1, ctx.last_plan()
    a, b = a.astype(np.float64), b.astype(np.float64)
    assert within(got, a @ b, np.abs(a) @ np.abs(b), 1044)


@pytest.mark.parametrize("k", [64, 512, 2048])
@pytest.mark.parametrize("positive", [False, True])
def test_errors_are_no_larger_than_the_fp32_instructions(ctx, split, k, positive):
    """2-norms against 64 bits over 512 x 512 results, uncut; and no drift to one side, which would add up over layers."""
    rng = np.random.default_rng(k)
    a, b = rng.standard_normal((512, k)).astype(np.float32), (rng.standard_normal((k, 512)) * 0.03).astype(np.float32)
    if positive:
        a, b = np.abs(a), np.abs(b)
    want = a.astype(np.float64) @ b.astype(np.float64)
    err, drift = {}, 0.0
    ctx.set_option("gemm_wavesplit", 0)
    try:
        for mode in (0, 6):
            split(mode)
            ctx.set_option("split_k", 1)
            got = product(ctx, a, b, True)
            err[mode] = np.linalg.norm(got - want) / np.linalg.norm(want)
            drift = float(np.sum((got - want) * np.sign(want)) / np.sum(np.abs(want)))
    finally:
        ctx.set_option("gemm_wavesplit", 1)
    assert err[6] <= err[0], err
    assert abs(drift) <= 2.0 ** -26, drift


@pytest.mark.parametrize("mode", [3, 6, 8, 9])
@pytest.mark.parametrize("transposed", [False, True])
def test_values_the_split_cannot_hold(ctx, split, mode, transposed):
    """Inf and NaN, the largest floats, sums that overflow, subnormals: as with the fp32 instruction."""
    rng = np.random.default_rng(11)
    a, b = rng.standard_normal((200, 100)).astype(np.float32), rng.standard_normal((100, 260)).astype(np.float32)
    a[3, 7], a[70, 99], a[130, 0] = np.inf, np.nan, -np.inf
    b[50, 5], b[99, 250] = np.inf, -np.inf
    a[5, :], b[:, 9] = 0, 0
    a[5, 2], b[2, 9] = np.finfo(np.float32).max, 1.0
    a[199, :], a[199, :2] = 0, 3e38  # (two products: the order of a longer sum would decide where it overflows)
    a[64, :] *= np.float32(1e-38)
    a[65, :] *= np.float32(1e-42)
    a[66, :] *= np.float32(1e-25)
    out = {}
    ctx.set_option("gemm_wavesplit", 0)
    try:
        for value in (0, mode):
            split(value)
            out[value] = product(ctx, a, b, transposed)
    finally:
        ctx.set_option("gemm_wavesplit", 1)
    assert ctx.last_plan()["tile"] == TILES[mode]
    want, got = out[0], out[mode]
    assert (np.isnan(want) == np.isnan(got)).all()
    assert (np.isposinf(want) == np.isposinf(got)).all() and (np.isneginf(want) == np.isneginf(got)).all()
    finite = np.isfinite(want)
    with np.errstate(all="ignore"):
        magnitudes = np.nan_to_num(np.abs(a.astype(np.float64)), posinf=0) @ np.nan_to_num(np.abs(b.astype(np.float64)), posinf=0)
    assert (np.abs(got.astype(np.float64) - want)[finite] <= (108 * 2.0 ** -23 * magnitudes + 2e-45 * 100)[finite]).all()


CONVS = [
    # n, cin, h, w, cout, kernel, stride, pad, dilation, group
    (3, 32, 8, 10, 70, 1, 1, 0, 1, 1),       # in place, pairs of pixels
    (2, 36, 7, 7, 64, 1, 1, 0, 1, 1),        # odd planes: a pixel at a time
    (5, 128, 9, 11, 130, 1, 2, 0, 1, 1),
    (2, 96, 13, 8, 40, 1, 3, 0, 1, 2),       # groups, a stride of 3
    (2, 64, 12, 12, 64, 1, 2, 0, 1, 1),      # even rows, stride 2
    (2, 16, 9, 14, 64, 3, 1, 1, 1, 1),
    (3, 64, 15, 11, 130, 3, 2, 1, 1, 1),
    (2, 24, 17, 19, 40, 5, 2, 2, 1, 2),      # 25 taps, ragged K, groups
    (2, 16, 20, 21, 24, 7, 1, 3, 1, 1),      # 49 taps
    (2, 20, 16, 16, 66, 3, 1, 2, 2, 1),      # dilated
]


@pytest.mark.parametrize("mode", [3, 4, 5, 6, 8, 9])
@pytest.mark.parametrize("shape", CONVS)
def test_convs(ctx, split, mode, shape):
    n, cin, h, w, cout, kernel, stride, pad, dil, group = shape
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal((n, cin, h, w)).astype(np.float32)
    wt, bias = rng.standard_normal((cout, cin // group, kernel, kernel)).astype(np.float32), rng.standard_normal(cout).astype(np.float32)
    ctx.set_option("conv3x3_winograd", 0)
    out = {}
    for value in (0, mode):
        split(value)
        y = H.conv(ctx, ctx.move_tensor(x), ctx.move_tensor(wt), ctx.move_tensor(bias), [dil, dil], group, None, [pad] * 4, [stride, stride],
                   epilogue="relu")
        out[value], plan = y.get_data(), ctx.last_plan()
    assert plan["tile"] == TILES[mode], plan
    y = H.conv(ctx, ctx.move_tensor(np.abs(x)), ctx.move_tensor(np.abs(wt)), ctx.move_tensor(np.abs(bias)), [dil, dil], group, None, [pad] * 4,
               [stride, stride])
    k = cin // group * kernel * kernel
    assert (np.abs(out[0].astype(np.float64) - out[mode]) <= 2 * (k + 8) * 2.0 ** -24 * y.get_data()).all()
    x[0, 1, h // 2, w // 2], x[n - 1, 0, 0, 0] = np.inf, np.nan   # what a padded tap must not touch stays clean
    for value in (0, mode):
        split(value)
        out[value] = H.conv(ctx, ctx.move_tensor(x), ctx.move_tensor(wt), ctx.move_tensor(bias), [dil, dil], group, None, [pad] * 4,
                            [stride, stride]).get_data()
    assert (np.isnan(out[0]) == np.isnan(out[mode])).all() and (np.isinf(out[0]) == np.isinf(out[mode])).all()


@pytest.mark.parametrize("shape", CONVS)
def test_convs_without_a_tile_of_that_size(ctx, split, shape):
    """There are no 256x128 tiles for convs: asked for them, a conv takes the fp32 instruction."""
    n, cin, h, w, cout, kernel, stride, pad, dil, group = shape
    rng = np.random.default_rng(sum(shape))
    x = rng.standard_normal((n, cin, h, w)).astype(np.float32)
    wt = rng.standard_normal((cout, cin // group, kernel, kernel)).astype(np.float32)
    ctx.set_option("conv3x3_winograd", 0)
    run = lambda x, wt: H.conv(ctx, ctx.move_tensor(x), ctx.move_tensor(wt), None, [dil, dil], group, None, [pad] * 4, [stride, stride]).get_data()
    split(0)
    want, magnitudes = run(x, wt), run(np.abs(x), np.abs(wt))
    split(7)
    got = run(x, wt)
    assert ctx.last_plan()["tile"] != TILES[7], ctx.last_plan()
    k = cin // group * kernel * kernel
    assert (np.abs(want.astype(np.float64) - got) <= 2 * (k + 8) * 2.0 ** -24 * magnitudes).all()


def test_one_image_keeps_its_bits(ctx, split):
    """A single image stays with the fp32 instruction; the same image in a batch agrees with it as sums in another order do."""
    rng = np.random.default_rng(4)
    x = rng.standard_normal((2, 256, 28, 28)).astype(np.float32)
    for cout, kernel in ((128, 1), (256, 3)):
        wt = ctx.move_tensor((rng.standard_normal((cout, 256, kernel, kernel)) * 0.03).astype(np.float32))
        out = {}
        for value in (0, 1):
            split(value)
            out[value] = H.conv(ctx, ctx.move_tensor(x[:1]), wt, pads=[kernel // 2] * 4).get_data()
        assert (out[0] == out[1]).all()
        both = H.conv(ctx, ctx.move_tensor(x), wt, pads=[kernel // 2] * 4).get_data()
        assert np.abs(both[:1] - out[0]).max() <= 1e-5 * np.abs(out[0]).max()


def test_a_geometry_first_met_while_recording(ctx, split):
    """The gathered form needs a tap table, which cannot be built then: the form that reads an LDS tile serves."""
    split(2)
    rng = np.random.default_rng(6)
    x, wt = ctx.move_tensor(rng.standard_normal((2, 72, 20, 24)).astype(np.float32)), ctx.move_tensor(rng.standard_normal((64, 72, 3, 3)).astype(np.float32))
    ctx.sync()
    ctx.graph_begin()
    y = H.conv(ctx, x, wt, pads=[1] * 4)
    form = ctx.last_plan()["form"]
    graph = ctx.graph_end()
    assert form == "conv 3x3, LDS tile", form
    for _ in range(3):
        ctx.graph_launch(graph)
        got = y.get_data()
        want = H.conv(ctx, x, wt, pads=[1] * 4)
        assert ctx.last_plan()["form"] == "conv, gathered taps", ctx.last_plan()
        assert np.abs(got - want.get_data()).max() <= 1e-5 * np.abs(got).max()
        want.dispose()
    ctx.graph_destroy(graph)


@pytest.mark.parametrize("shape,pays", [((118, 192, 8, 8, 320, 3, 2), False), ((13, 264, 11, 47, 192, 3, 1), False),
                                        ((64, 128, 28, 28, 256, 3, 2), True)])
def test_gathered_taps_pay_where_128_channels_share_them(ctx, split, shape, pays):
    """Where no tile of 128 channels is planned the fp32 instruction serves, bit for bit; elsewhere the other one is taken."""
    n, cin, h, w, cout, kernel, stride = shape
    rng = np.random.default_rng(sum(shape))
    x = ctx.move_tensor(rng.standard_normal((n, cin, h, w)).astype(np.float32))
    wt = ctx.move_tensor(rng.standard_normal((cout, cin, kernel, kernel)).astype(np.float32))
    out, plans = [], []
    for value in (0, 1):
        split(value)
        out.append(H.conv(ctx, x, wt, pads=[1] * 4, strides=[stride, stride]).get_data())
        plans.append(ctx.last_plan())
    assert (plans[0] == plans[1] and (out[0] == out[1]).all()) == (not pays), plans


# (us, the form that was taken before / the one that is)
@pytest.mark.parametrize("shape,form", [((4, 512, 45, 63, 160), "F(2x2,3x3)"), ((2, 832, 63, 63, 192), "F(2x2,3x3)"),   # rows 141 / 100, 149 / 105
                                        ((13, 336, 19, 91, 416), "F(2x2,3x3)"),                                        # gathered taps 447 / 293
                                        ((32, 128, 28, 28, 128), "LDS tile"), ((32, 256, 14, 14, 256), "F(2x2,3x3)")])
def test_3x3_convs_take_the_form_of_the_least_estimate(ctx, split, shape, form):
    n, cin, h, w, cout = shape
    rng = np.random.default_rng(sum(shape))
    x = ctx.move_tensor(rng.standard_normal((n, cin, h, w)).astype(np.float32))
    wt = ctx.move_tensor(rng.standard_normal((cout, cin, 3, 3)).astype(np.float32))
    y = H.conv(ctx, x, wt, pads=[1] * 4)
    assert form in ctx.last_plan()["form"], ctx.last_plan()
    got = y.get_data()
    ctx.set_option("conv3x3_winograd", 0)
    split(0)
    want = H.conv(ctx, x, wt, pads=[1] * 4).get_data()
    assert np.abs(got.astype(np.float64) - want).max() <= 1e-5 * np.abs(want).max()


def test_a_product_short_of_blocks_stays_with_the_fp32_instruction(ctx, split):
    """223x2292x1272: 22.6 us in 64x64 tiles whose K four groups share, 17.6 in blocks of 32x32."""
    a, b = ctx.move_tensor(np.ones((223, 1272), np.float32)), ctx.move_tensor(np.ones((1272, 2292), np.float32))
    assert (H.gemm(ctx, a, b).get_data() == 1272).all()
    assert ctx.last_plan()["tile"] == "32x32", ctx.last_plan()


def test_gathered_taps_of_a_full_round_of_tiles_and_a_few(ctx, split):
    """28 images 672 -> 544, stride 2, on 18x25: 256 of 260 128x64 tiles whole and four in 32 chunks each 263 us, 128x128 tiles 191."""
    rng = np.random.default_rng(19)
    x = ctx.move_tensor(rng.standard_normal((28, 672, 18, 25)).astype(np.float32))
    wt = ctx.move_tensor(rng.standard_normal((544, 672, 3, 3)).astype(np.float32))
    got = H.conv(ctx, x, wt, pads=[1] * 4, strides=[2, 2]).get_data()
    assert ctx.last_plan()["tile"] == "128x128", ctx.last_plan()
    split(0)
    want = H.conv(ctx, x, wt, pads=[1] * 4, strides=[2, 2]).get_data()
    assert np.abs(got.astype(np.float64) - want).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("shape,residual,small", [((42, 96, 15, 77, 512, 1), True, True), ((42, 96, 15, 77, 512, 1), False, True), ((8, 192, 28, 28, 512, 2), True, True),
                                                  ((64, 128, 28, 28, 512, 1), True, True), ((64, 128, 28, 28, 512, 1), False, True), ((64, 208, 28, 28, 512, 1), True, False),
                                                  ((88, 128, 28, 28, 512, 1), True, False)])
def test_1x1_convs_of_a_short_k_take_small_tiles(ctx, split, shape, residual, small):
    """In place, a pixel at a time and with stride 2; what bounds them is the results and the residual."""
    n, cin, h, w, cout, stride = shape
    rng = np.random.default_rng(17)
    x = ctx.move_tensor(rng.standard_normal((n, cin, h, w)).astype(np.float32))
    wt = ctx.move_tensor(rng.standard_normal((cout, cin, 1, 1)).astype(np.float32))
    r = ctx.move_tensor(rng.standard_normal((n, cout, h // stride, w // stride)).astype(np.float32)) if residual else None
    out = []
    for value in (0, 1):
        split(value)
        out.append(H.conv(ctx, x, wt, residual=r, strides=[stride, stride]).get_data())
    assert (ctx.last_plan()["tile"] == "64x64") == small, ctx.last_plan()
    assert not (out[0] == out[1]).all()
    assert np.abs(out[0].astype(np.float64) - out[1]).max() <= 1e-5 * np.abs(out[0]).max()


@pytest.mark.parametrize("n,cin,h,w,cout,kernel,stride", [(42, 96, 15, 77, 128, 1, 1), (5, 128, 28, 28, 512, 1, 1), (3, 160, 14, 14, 320, 1, 1), (2, 256, 23, 31, 96, 1, 2),
                                                          (4, 512, 45, 63, 160, 3, 1), (12, 128, 34, 39, 128, 3, 1), (6, 128, 30, 30, 128, 3, 2)])
def test_a_residual_does_not_decide_the_form(ctx, n, cin, h, w, cout, kernel, stride):
    """Conv with bias, residual and Relu in one launch has the bits of the three nodes."""
    rng = np.random.default_rng(n + cin + h)
    pads = [kernel // 2] * 4
    x, wt = rng.standard_normal((n, cin, h, w)).astype(np.float32), rng.standard_normal((cout, cin, kernel, kernel)).astype(np.float32)
    x, wt, b = ctx.move_tensor(x), ctx.move_tensor(wt), ctx.move_tensor(rng.standard_normal(cout).astype(np.float32))
    y = H.conv(ctx, x, wt, b, pads=pads, strides=[stride, stride])
    r = ctx.move_tensor(rng.standard_normal(y.dims).astype(np.float32))
    want = H.unary(ctx, "Relu", H.binary(ctx, "Add", y, r)).get_data()
    got = H.conv(ctx, x, wt, b, pads=pads, strides=[stride, stride], residual=r, epilogue="relu").get_data()
    assert (got == want).all()


ROWS = [
    # n, c, h, w, cout, pads: ragged tiles and channels, tiles over several images, unequal and wide pads, wide rows
    (2, 16, 8, 9, 64, [1, 1, 1, 1]),
    (3, 64, 15, 13, 70, [1, 1, 1, 1]),
    (9, 48, 5, 5, 130, [1, 1, 1, 1]),
    (2, 32, 11, 7, 64, [0, 0, 0, 0]),
    (3, 80, 10, 12, 128, [2, 0, 1, 2]),
    (2, 32, 6, 78, 64, [1, 1, 1, 1]),
    (20, 16, 3, 3, 64, [1, 1, 1, 1]),
]


@pytest.mark.parametrize("mode,chunks", [(3, 1), (4, 1), (4, 2), (2, -1)])
@pytest.mark.parametrize("shape", ROWS)
def test_rows_of_3x3_convs(ctx, split, mode, chunks, shape):
    """Input rows in LDS, weights laid out in parts; kept per buffer when the caller vouches for them, until it is written to."""
    n, c, h, w, cout, pads = shape
    rng = np.random.default_rng(sum(shape[:5]))
    x = rng.standard_normal((n, c, h, w)).astype(np.float32)
    wt, bias = rng.standard_normal((cout, c, 3, 3)).astype(np.float32), rng.standard_normal(cout).astype(np.float32)
    tx, tw, tb = (ctx.move_tensor(v) for v in (x, wt, bias))
    ctx.set_option("conv3x3_winograd", 0)
    split(0)
    plain = H.conv(ctx, tx, tw, tb, pads=pads)
    r = rng.standard_normal(plain.dims).astype(np.float32)
    tr = ctx.move_tensor(r)
    want = np.maximum(plain.get_data().astype(np.float64) + r, 0)
    bound = 2 * (9 * c + 8) * 2.0 ** -24 * (H.conv(ctx, *(ctx.move_tensor(np.abs(v)) for v in (x, wt, bias)), pads=pads).get_data() + np.abs(r))
    split(mode)
    ctx.set_option("split_k", chunks)
    for constant in (False, True, True):
        got = H.conv(ctx, tx, tw, tb, pads=pads, epilogue="relu", residual=tr, constant_weights=constant)
        plan = ctx.last_plan()
        assert plan["form"] == "conv 3x3, LDS tile" and plan["tile"] in ("128x128", "64x128"), plan
        assert (np.abs(got.get_data() - want) <= bound).all()
    tw.set_data(2 * wt)
    again = H.conv(ctx, tx, tw, None, pads=pads, constant_weights=True).get_data()
    assert (np.abs(again - 2 * (plain.get_data().astype(np.float64) - bias.reshape(1, -1, 1, 1))) <= 4 * bound + 1e-5).all()
    x[0, c - 1, h // 2, w // 2], x[n - 1, 0, 0, 0] = np.inf, np.nan
    tx.set_data(x)
    out = {}
    for value in (0, mode):
        split(value)
        out[value] = H.conv(ctx, tx, tw, tb, pads=pads).get_data()
    assert (np.isnan(out[0]) == np.isnan(out[mode])).all() and (np.isinf(out[0]) == np.isinf(out[mode])).all()


def test_rows_while_recording(ctx, split):
    """Weights laid out while a graph is recorded belong to it; those kept from before are used by it."""
    rng = np.random.default_rng(8)
    x, wt = ctx.move_tensor(rng.standard_normal((4, 64, 20, 24)).astype(np.float32)), ctx.move_tensor(rng.standard_normal((64, 64, 3, 3)).astype(np.float32))
    want = H.conv(ctx, x, wt, pads=[1] * 4).get_data()
    for warm in (False, True):
        if warm:
            H.conv(ctx, x, wt, pads=[1] * 4, constant_weights=True).dispose()
        ctx.sync()
        ctx.graph_begin()
        y = H.conv(ctx, x, wt, pads=[1] * 4, constant_weights=True)
        graph = ctx.graph_end()
        for _ in range(3):
            ctx.graph_launch(graph)
            assert (y.get_data() == want).all()
            other = H.conv(ctx, x, wt, pads=[1] * 4)
            assert (other.get_data() == want).all()
            other.dispose()
        ctx.graph_destroy(graph)


def test_recorded_weights_outlive_another_size(ctx, split):
    """One weight, two sizes of input that take two forms: what a recorded run reads stays while the other size runs."""
    rng = np.random.default_rng(10)
    wt = ctx.move_tensor(rng.standard_normal((128, 128, 3, 3)).astype(np.float32))
    large, small = (ctx.move_tensor(rng.standard_normal((n, 128, s, s)).astype(np.float32)) for n, s in ((4, 32), (2, 10)))
    run = lambda x: H.conv(ctx, x, wt, pads=[1] * 4, constant_weights=True)
    want, forms = [], []
    for x in (large, small):
        want.append(H.conv(ctx, x, wt, pads=[1] * 4).get_data())
        forms.append(ctx.last_plan()["form"])
    assert forms[0] != forms[1], forms
    for recorded, other, a, b in ((large, small, *want), (small, large, *want[::-1])):
        run(recorded).dispose()
        ctx.sync()
        ctx.graph_begin()
        y = run(recorded)
        graph = ctx.graph_end()
        for _ in range(3):
            z = run(other)
            # (blocks that went back to the pool are written over)
            junk = [ctx.move_tensor(np.full(elements, 7.0, np.float32)) for elements in (221184, 262144) * 4]
            ctx.graph_launch(graph)
            assert (y.get_data() == a).all() and (z.get_data() == b).all()
            for t in junk + [z]:
                t.dispose()
        ctx.graph_destroy(graph)


@pytest.mark.parametrize("shift", [-120, -112, -100])
def test_rows_of_tiny_elements(ctx, split, shift):
    """Elements whose last part does not fit bfloat16 leave tiny sums, which are added up again, also against large partners."""
    rng = np.random.default_rng(11)
    a = (rng.uniform(1, 2, (256, 512)) * 2.0 ** shift).astype(np.float32)
    b = (rng.uniform(1, 2, (512, 256)) * 2.0 ** 40).astype(np.float32)
    split(3)
    got = product(ctx, a, b, False)
    assert ctx.last_plan()["tile"] == "128x128"
    a, b = a.astype(np.float64), b.astype(np.float64)
    assert within(got, a @ b, a @ b, 512)


# exponents of the tiny operand and of its partners: some bits lost, all lost, subnormal floats; results from 2^-128 to 2^-17
TINY = [(-112, 40), (-118, 12), (-118, 100), (-126, 64), (-126, 100), (-135, 100), (-140, 12), (-140, 100)]


def uniform(rng, shape, exponent):
    return (rng.uniform(1, 2, shape) * 2.0 ** exponent).astype(np.float32)


def sums_hold(got, want, magnitudes, k):
    """As `within`, down to the least float there is."""
    return (np.abs(got - want) <= (k + 8) * 2.0 ** -24 * magnitudes + k * 2.0 ** -149).all()


@pytest.mark.parametrize("mode", [3, 6, 7, 8, 9])
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("tiny,partner", TINY)
def test_tiny_elements(ctx, split, mode, transposed, tiny, partner):
    """Elements that bfloat16 parts hold in part or not at all, as the left and as the right operand, nothing else in the tile."""
    rng = np.random.default_rng(11)
    a, b = uniform(rng, (256, 144), tiny), uniform(rng, (144, 256), partner)
    split(mode)
    ctx.set_option("gemm_wavesplit", 0)
    try:
        for l, r in ((a, b), (np.ascontiguousarray(b.T), np.ascontiguousarray(a.T))):
            got = product(ctx, l, r, transposed)
            assert ctx.last_plan()["tile"] == TILES[mode]
            want = l.astype(np.float64) @ r.astype(np.float64)
            assert sums_hold(got, want, want, 144)
    finally:
        ctx.set_option("gemm_wavesplit", 1)


@pytest.mark.parametrize("mode", [3, 9])
@pytest.mark.parametrize("chunks", [1, 3])
@pytest.mark.parametrize("partner", [100, 30, -3])
def test_tiny_elements_among_others(ctx, split, mode, chunks, partner):
    """One of them in a row of ordinary elements: it counts where its partner lifts it, and every sum is far above 2^-60."""
    rng = np.random.default_rng(12)
    a, b = uniform(rng, (256, 192), -30), uniform(rng, (192, 256), -20)
    for at in (0, 100, 191):   # (one in each chunk)
        a[:, at], b[at] = uniform(rng, 256, -126), uniform(rng, 256, partner)
    split(mode)
    ctx.set_option("split_k", chunks)
    got = product(ctx, a, b, False)
    assert ctx.last_plan()["tile"] == TILES[mode] and ctx.last_plan()["split"] == chunks
    a, b = a.astype(np.float64), b.astype(np.float64)
    assert sums_hold(got, a @ b, a @ b, 192)


# one slab, a ragged last one, an odd and an even number of slabs; edges in both directions; cut along K
@pytest.mark.parametrize("mode", sorted(TILES))
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("m,n,k,chunks", [(64, 64, 16, 1), (65, 132, 44, 1), (129, 68, 64, 1), (257, 260, 76, 1), (100, 196, 244, 3)])
def test_tiles_done_again(ctx, split, mode, transposed, m, n, k, chunks):
    rng = np.random.default_rng(m + n + k)
    a, b = rng.standard_normal((m, k)).astype(np.float32) * np.float32(2.0 ** -120), rng.standard_normal((k, n)).astype(np.float32) * np.float32(2.0 ** 120)
    bias = rng.standard_normal(n).astype(np.float32)
    split(mode)
    ctx.set_option("gemm_wavesplit", 0)
    ctx.set_option("split_k", chunks)
    try:
        got = product(ctx, a, b, transposed, bias)
    finally:
        ctx.set_option("gemm_wavesplit", 1)
    assert ctx.last_plan()["tile"] == TILES[mode], ctx.last_plan()
    a, b = a.astype(np.float64), b.astype(np.float64)
    assert within(got, a @ b + bias, np.abs(a) @ np.abs(b) + np.abs(bias), k)


@pytest.mark.parametrize("kind", ["gemm", "rows", "taps", "pixels"])
def test_tiles_done_again_cost_little_more_than_the_fp32_instruction(ctx, split, kind):
    """A NaN that reaches every tile: both instructions one after the other, each at its own pace (with loads a
    single element at a time it was 3.5 to 5.5 times)."""
    rng = np.random.default_rng(15)
    if kind == "gemm":
        a, b = rng.standard_normal((2048, 2048)).astype(np.float32), rng.standard_normal((2048, 2048)).astype(np.float32)
        a[:, 5] = np.nan
        ta, tb = ctx.move_tensor(a), ctx.move_tensor(b)
        run = lambda: H.gemm(ctx, ta, tb, trans_b=1)
    else:
        cin, cout, size, kernel, stride = {"rows": (128, 128, 28, 3, 1), "taps": (128, 128, 56, 3, 2), "pixels": (256, 512, 28, 1, 2)}[kind]
        x, w = rng.standard_normal((32, cin, size, size)).astype(np.float32), rng.standard_normal((cout, cin, kernel, kernel)).astype(np.float32)
        w[::8] = np.nan
        tx, tw = ctx.move_tensor(x), ctx.move_tensor(w)
        ctx.set_option("conv3x3_winograd", 0)
        run = lambda: H.conv(ctx, tx, tw, pads=[kernel // 2] * 4, strides=[stride, stride], constant_weights=True)
    best = {}
    for value in (0, 1):
        split(value)
        run().dispose()
        times = []
        for _ in range(5):
            ctx.event_record(0)
            for _ in range(5):
                run().dispose()
            ctx.event_record(1)
            ctx.sync()
            times.append(ctx.event_elapsed_ms(0, 1))
        best[value] = min(times)
    assert best[1] <= 2.8 * best[0], best


@pytest.mark.parametrize("mode", [3, 4])
@pytest.mark.parametrize("kernel,stride", [(3, 1), (3, 2), (1, 1), (1, 2)])
@pytest.mark.parametrize("tiny,partner", TINY)
def test_tiny_elements_of_convs(ctx, split, mode, kernel, stride, tiny, partner):
    """The same in the input and in the weights (which the 3x3 form lays out beforehand)."""
    rng = np.random.default_rng(13)
    split(mode)
    ctx.set_option("conv3x3_winograd", 0)
    for ex, ew in ((tiny, partner), (partner, tiny)):
        x, w = uniform(rng, (2, 32, 12, 12), ex), uniform(rng, (128, 32, kernel, kernel), ew)
        tw = ctx.move_tensor(w)
        pad = kernel // 2
        padded = np.pad(x.astype(np.float64), ((0, 0), (0, 0), (pad, pad), (pad, pad)))
        windows = np.lib.stride_tricks.sliding_window_view(padded, (kernel, kernel), (2, 3))[:, :, ::stride, ::stride]
        want = np.einsum("ncyxij,ocij->noyx", windows, w.astype(np.float64))
        for constant in (False, True, True):
            got = H.conv(ctx, ctx.move_tensor(x), tw, pads=[pad] * 4, strides=[stride, stride], constant_weights=constant).get_data()
            assert ctx.last_plan()["tile"] == TILES[mode]
            assert sums_hold(got, want, want, 32 * kernel * kernel)


@pytest.mark.parametrize("mode,form", [(1, 1), (3, 1), (6, 3)])
def test_transformed_convs_do_not_see_what_the_pool_held(ctx, split, mode, form):
    """60 (20) tiles in rows of 64 (32): what lies behind them is not another matrix's rest."""
    rng = np.random.default_rng(14)
    n, c, h, w = 5, 512, 6, 8
    x = ctx.move_tensor(rng.standard_normal((n, c, h, w)).astype(np.float32))
    wt = ctx.move_tensor((rng.standard_normal((c, c, 3, 3)) * 0.02).astype(np.float32))
    split(mode)
    ctx.set_option("conv3x3_winograd", form)
    positions, pitch = (16, 64) if form == 1 else (36, 32)
    elements = positions * c * pitch
    out = []
    for junk in (np.zeros(elements, np.float32), np.full(elements, np.nan, np.float32), np.full(elements, 5, np.int32)):
        held = [ctx.move_tensor(junk) for _ in range(4)]
        for t in held:
            t.dispose()
        y = H.conv(ctx, x, wt, pads=[1] * 4)
        assert "transforms" in ctx.last_plan()["form"], ctx.last_plan()
        out.append(y.get_data())
        y.dispose()
    assert (out[0] == out[1]).all() and (out[0] == out[2]).all()


@pytest.mark.parametrize("mode", sorted(TILES))
@pytest.mark.parametrize("n", [4, 70, 131, 132, 250])
def test_columns_beside_a_matrix_stay_out(ctx, split, mode, n):
    """B as the first columns of a wider buffer: what lies beside them changes no bit, also where a tile reads it."""
    rng = np.random.default_rng(n)
    m, k, ld = 96, 80, 264
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((k, ld)).astype(np.float32)
    ta, y = ctx.move_tensor(a), ctx.empty_tensor([m, n])
    split(mode)
    ctx.set_option("gemm_wavesplit", 0)
    out = []
    try:
        for beside in (0.0, np.nan, 1e-40):
            b[:, n:] = beside
            tb = ctx.move_tensor(b)
            capi.call("wdh_gemm_ex", ta.handle, tb.handle, 0, y.handle, 1, m, n, k, 0, k, 1, 0, ld, 1, 0, 0, 1.0, 1.0, 0, 0, m * n, n)
            out.append(y.get_data())
    finally:
        ctx.set_option("gemm_wavesplit", 1)
    a, b = a.astype(np.float64), b[:, :n].astype(np.float64)
    assert within(out[0], a @ b, np.abs(a) @ np.abs(b), k)
    assert (out[0] == out[1]).all() and (out[0] == out[2]).all()


@pytest.mark.parametrize("mode", [m for m in sorted(TILES) if m != 7])
def test_pixels_past_the_last_stay_in_their_channel(ctx, split, mode):
    """A 1x1 conv's surplus columns repeat the last pixels: the next channel's first one, a NaN, changes no bit of their tile."""
    rng = np.random.default_rng(18)
    x, wt = rng.standard_normal((2, 128, 10, 10)).astype(np.float32), ctx.move_tensor(rng.standard_normal((128, 128, 1, 1)).astype(np.float32))
    split(mode)
    out = []
    for value in (0.5, np.nan):
        x[1, 5, 0, 0] = value
        out.append(H.conv(ctx, ctx.move_tensor(x), wt).get_data())
        assert ctx.last_plan()["tile"] == TILES[mode] and "in place" in ctx.last_plan()["form"], ctx.last_plan()
    assert np.isnan(out[1][1, :, 0, 0]).all()
    assert (out[0][1, :, 9, 2:] == out[1][1, :, 9, 2:]).all()  # (pixels 192 to 199 of 200)


def test_groups_that_fill_the_chip(ctx, split):
    """The projections of an attention block as one launch of 64x64 tiles; ragged rows and columns, one weight k-contiguous by shape."""
    rng = np.random.default_rng(9)
    for t, d, n in ((384, 768, 768), (509, 512, 516), (256, 768, 772)):
        x = rng.standard_normal((t, d)).astype(np.float32)
        x[t - 1, 5] = np.inf if n == 772 else 1.0
        ws = [(rng.standard_normal((d, n)).astype(np.float32), rng.standard_normal(n).astype(np.float32)) for _ in range(3)]
        tx = ctx.move_tensor(x)
        args = [(tx, ctx.move_tensor(w), ctx.move_tensor(b)) for w, b in ws]
        out = {}
        for value in (0, 1):
            split(value)
            out[value] = [y.get_data() for y in H.linear_group(ctx, args)]
            assert ctx.last_plan()["tile"] == ("64x64" if value else "32x32"), ctx.last_plan()
        rows = slice(0, t - 1)
        for (w, b), y0, y1 in zip(ws, out[0], out[1]):
            a64, w64 = x[rows].astype(np.float64), w.astype(np.float64)
            assert within(y1[rows], a64 @ w64 + b, np.abs(a64) @ np.abs(w64) + np.abs(b), d)
            assert (np.isfinite(y0) == np.isfinite(y1)).all()
