"""Depthwise convolutions (one input channel per group) on the GPU against the oracle."""
import numpy as np
import pytest

from oracle import ref
from util import assert_bit_exact
from webdnn_amd import hostops as H

pytestmark = pytest.mark.gpu

CASES = [
    # n, c, multiplier, h, w, kernel, pads, strides, dilations, rows x columns of a thread
    (2, 16, 1, 9, 9, (3, 3), [1, 1, 1, 1], [1, 1], [1, 1], "1x1"),        # a small launch of ragged rows: a thread per output
    (1, 3, 1, 1, 1, (3, 3), [1, 1, 1, 1], [1, 1], [1, 1], "1x1"),         # a single cell, every other tap in the padding
    (3, 5, 1, 7, 7, (3, 3), [1, 1, 1, 1], [1, 1], [1, 1], "1x1"),         # planes packed into wavefronts
    (16, 168, 1, 7, 7, (3, 3), [1, 1, 1, 1], [1, 1], [1, 1], "1x4"),      # and as ragged column tiles
    (24, 60, 1, 9, 9, (3, 3), [0, 1, 3, 1], [1, 1], [1, 1], "1x1"),       # the last size of a thread per output
    (28, 58, 1, 9, 9, (3, 3), [0, 1, 3, 1], [1, 1], [1, 1], "1x4"),       # whole rows of taps in the padding
    (2, 3, 1, 4, 4, (3, 3), [1, 1, 1, 1], [1, 1], [1, 1], "1x4"),
    (16, 64, 1, 36, 40, (3, 3), [1, 1, 1, 1], [1, 1], [1, 1], "1x4"),     # whole 16-byte tiles
    (8, 320, 1, 32, 48, (3, 3), [1, 1, 1, 1], [1, 1], [1, 1], "1x4"),     # the last size before four rows a thread
    (8, 352, 1, 32, 48, (3, 3), [1, 1, 1, 1], [1, 1], [1, 1], "4x4"),
    (8, 360, 1, 33, 46, (3, 3), [1, 1, 1, 1], [1, 1], [1, 1], "4x4"),     # three of the last four rows and two of four columns empty
    (8, 320, 1, 66, 95, (3, 3), [1, 1, 1, 1], [2, 2], [1, 1], "2x4"),     # stride 2, odd rows
    (2, 8, 1, 11, 14, (3, 3), [0, 1, 1, 0], [2, 2], [1, 1], "1x1"),       # unequal pads
    (2, 8, 1, 12, 13, (3, 3), [3, 1, 2, 3], [1, 1], [1, 1], "1x1"),       # whole rows in the padding
    (64, 80, 1, 11, 14, (3, 3), [0, 1, 1, 0], [2, 2], [1, 1], "1x4"),     # the same as tiles
    (16, 60, 1, 12, 13, (3, 3), [3, 1, 2, 3], [1, 1], [1, 1], "1x4"),
    (2, 6, 1, 15, 18, (5, 5), [2, 2, 2, 2], [1, 1], [1, 1], "1x1"),
    (4, 160, 1, 48, 50, (5, 5), [2, 2, 2, 2], [1, 1], [1, 1], "1x4"),
    (4, 424, 1, 48, 50, (5, 5), [2, 2, 2, 2], [1, 1], [1, 1], "4x4"),     # four rows a thread, 5x5
    (4, 424, 1, 46, 49, (5, 5), [2, 2, 2, 2], [1, 1], [1, 1], "4x4"),     # two of the last four rows and three of four columns empty
    (2, 6, 1, 15, 18, (5, 5), [2, 2, 2, 2], [2, 2], [1, 1], "1x1"),
    (4, 330, 1, 48, 49, (5, 5), [2, 2, 2, 2], [2, 2], [1, 1], "1x4"),
    (8, 392, 1, 48, 49, (5, 5), [2, 2, 2, 2], [2, 2], [1, 1], "2x4"),     # two rows a thread
    (8, 392, 1, 46, 49, (5, 5), [2, 2, 2, 2], [2, 2], [1, 1], "2x4"),     # and one of the last two empty
    (2, 4, 3, 10, 11, (3, 3), [1, 1, 1, 1], [1, 1], [1, 1], "1x1"),       # three output channels per input channel
    (4, 100, 3, 10, 12, (3, 3), [1, 1, 1, 1], [1, 1], [1, 1], "1x4"),
    (2, 3, 16, 14, 9, (3, 3), [1, 1, 1, 1], [1, 1], [1, 1], "1x1"),       # as many as this form takes
    (2, 3, 16, 14, 12, (3, 3), [1, 1, 1, 1], [1, 1], [1, 1], "1x4"),
    (2, 4, 1, 10, 11, (3, 3), [2, 2, 2, 2], [1, 1], [2, 2], "1x1"),       # dilation: the general kernel
    (2, 4, 2, 10, 11, (7, 2), [3, 0, 3, 1], [2, 3], [1, 1], "1x1"),
]


@pytest.mark.parametrize("case", CASES)
def test_depthwise_conv(ctx, case):
    n, c, mult, h, w, (kh, kw), pads, strides, dil, tile = case
    rng = np.random.default_rng(1000 * c + 10 * h + w)
    X = rng.standard_normal((n, c, h, w)).astype(np.float32)
    W = rng.standard_normal((c * mult, 1, kh, kw)).astype(np.float32)
    B = rng.standard_normal(c * mult).astype(np.float32)
    tx, tw, tb = ctx.move_tensor(X), ctx.move_tensor(W), ctx.move_tensor(B)
    got = H.conv(ctx, tx, tw, tb, dil, c, None, pads, strides).get_data()
    want = ref.conv(X, W, B, dil, c, None, pads, strides)
    # a chain of kh*kw fp32 products and the bias: each of at most 2^-24 of the sum of magnitudes so far
    bound = (kh * kw + 2) * 2.0 ** -24 * ref.conv(np.abs(X), np.abs(W), np.abs(B), dil, c, None, pads, strides)
    plan, (rows, cols) = ctx.last_plan(), map(int, tile.split("x"))
    assert plan["form"] == "conv, depthwise" and plan["tile"] == tile, plan
    assert plan["whole_tiles"] == n * c * mult * -(-want.shape[2] // rows) * -(-want.shape[3] // cols)
    assert got.shape == want.shape
    assert np.all(np.abs(got.astype(np.float64) - want) <= bound)
    R = rng.standard_normal(want.shape).astype(np.float32)
    fused = H.conv(ctx, tx, tw, tb, dil, c, None, pads, strides, "relu", ctx.move_tensor(R)).get_data()
    assert_bit_exact(fused, np.maximum(got + R, 0) + 0.0, "depthwise conv + residual + relu")


def test_depthwise_conv_keeps_nan_and_inf_in_place(ctx):
    X, W = np.ones((1, 2, 12, 13), np.float32), np.ones((2, 1, 3, 3), np.float32)
    X[0, 0, 5, 6], X[0, 1, 0, 12] = np.nan, np.inf
    got = H.conv(ctx, ctx.move_tensor(X), ctx.move_tensor(W), None, None, 2, None, [1, 1, 1, 1]).get_data()
    assert_bit_exact(got, ref.conv(X, W, None, None, 2, None, [1, 1, 1, 1]), "NaN and Inf")


# where the matrix tiles are the faster form (us, the pass over memory against the tiles): a kernel as large as its plane
# 185 / 30, a long chain of taps for few outputs 12.4 / 9.3, many outputs an input channel 143 / 91 and 465 / 215
@pytest.mark.parametrize("n,c,mult,hw,k,pad,dil", [(1, 256, 1, 28, 28, 0, 1), (1, 1, 1, 28, 11, 0, 1), (8, 64, 16, 56, 3, 2, 2), (8, 64, 16, 56, 7, 3, 1)])
def test_depthwise_convs_that_stay_with_the_matrix_tiles(ctx, n, c, mult, hw, k, pad, dil):
    rng = np.random.default_rng(hw + k)
    X = rng.standard_normal((n, c, hw, hw)).astype(np.float32)
    W = rng.standard_normal((c * mult, 1, k, k)).astype(np.float32)
    got = H.conv(ctx, ctx.move_tensor(X), ctx.move_tensor(W), None, [dil, dil], c, None, [pad] * 4).get_data()
    assert ctx.last_plan()["form"].startswith("conv, gathered taps"), ctx.last_plan()
    want = ref.conv(X, W, None, [dil, dil], c, None, [pad] * 4)
    bound = (k * k + 2) * 2.0 ** -24 * ref.conv(np.abs(X), np.abs(W), None, [dil, dil], c, None, [pad] * 4)
    assert np.all(np.abs(got.astype(np.float64) - want) <= bound)


def test_large_kernels_add_up_by_rows(ctx):
    rng = np.random.default_rng(31)
    X, W = rng.standard_normal((1, 128, 28, 28)).astype(np.float32), rng.standard_normal((128, 1, 31, 31)).astype(np.float32)
    got = H.conv(ctx, ctx.move_tensor(X), ctx.move_tensor(W), None, None, 128, None, [15] * 4).get_data()
    assert ctx.last_plan()["form"] == "conv, depthwise"
    wide = np.pad(X[0].astype(np.float64), ((0, 0), (15, 15), (15, 15)))
    want = np.zeros((128, 28, 28))
    for ky in range(31):
        for kx in range(31):
            want += W[:, :, ky, kx].astype(np.float64)[:, :, None] * wide[:, ky:ky + 28, kx:kx + 28]
    # 31 + 31 additions, each of a rounding error of 2^-24 / sqrt(3) of a sum no larger than the result, that add up as
    # squares: 2.7e-7 (one chain of 961 taps measured 4.1e-7)
    assert np.linalg.norm(got[0] - want) <= np.sqrt(62 / 3) * 2.0 ** -24 * np.linalg.norm(want)


def test_a_geometry_first_met_while_recording(ctx):
    """The matrix tiles read a table that cannot be built while a graph is recorded; the depthwise form needs none."""
    rng = np.random.default_rng(1)
    X, W = rng.standard_normal((1, 6, 23, 23)).astype(np.float32), rng.standard_normal((6, 1, 23, 23)).astype(np.float32)
    tx, tw = ctx.move_tensor(X), ctx.move_tensor(W)
    ctx.sync()
    ctx.graph_begin()
    y = H.conv(ctx, tx, tw, None, None, 6)
    graph = ctx.graph_end()
    assert ctx.last_plan()["form"] == "conv, depthwise"
    want, magnitude = ref.conv(X, W, None, None, 6), ref.conv(np.abs(X), np.abs(W), None, None, 6)
    for _ in range(3):
        ctx.graph_launch(graph)
        assert np.all(np.abs(y.get_data().astype(np.float64) - want) <= 531 * 2.0 ** -24 * magnitude)
    ctx.graph_destroy(graph)
