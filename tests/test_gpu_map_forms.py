"""Reductions over an inner axis, squares and Sigmoid on the GPU, where they take forms of their own."""
import numpy as np
import pytest

from oracle import ref
from util import ulp_diff
from webdnn_amd import capi
from webdnn_amd import hostops as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,axis", [((3, 31, 5), 1), ((2, 32, 7), 1), ((2, 500, 17), 1), ((1, 33, 16), 1), ((40, 129, 500), 1),
                                        ((300, 63, 255), 1), ((7, 1, 11), 1), ((3, 7, 300), 1), ((3, 8, 300), 1), ((3, 9, 300), 1), ((4, 5, 70000), 1), ((1, 71, 66000), 1)])
def test_mean_over_an_inner_axis(ctx, shape, axis):
    x = np.random.default_rng(sum(shape)).standard_normal(shape).astype(np.float32)
    got = H.reduce_mean(ctx, ctx.move_tensor(x), [axis], 0).get_data()
    want = x.astype(np.float64).sum(axis) / shape[axis]
    # sums in double whatever their order: one rounding to fp32, and a sum's double error under cancellation
    slack = shape[axis] * 2.0 ** -52 * np.abs(x.astype(np.float64)).mean(axis)
    assert (np.abs(got - want) <= 2.0 ** -24 * np.abs(want) * 1.0001 + slack).all()


def test_square_is_the_rounded_double_product(ctx):
    rng = np.random.default_rng(9)
    x = np.concatenate([rng.standard_normal(4099) * 10.0 ** rng.integers(-30, 19, 4099),
                        [0.0, -0.0, np.inf, -np.inf, np.nan, 1e-45, 3e38]]).astype(np.float32)
    with np.errstate(over="ignore", under="ignore"):
        want = (x.astype(np.float64) * x.astype(np.float64)).astype(np.float32)
    two = ctx.move_tensor(np.array([2.0], np.float32))
    got = H.binary(ctx, "Pow", ctx.move_tensor(x), two).get_data()
    assert (got.view(np.uint32) == want.view(np.uint32))[~np.isnan(want)].all() and np.isnan(got[np.isnan(want)]).all()
    mixed = np.where(np.arange(x.size) % 3 == 0, 2.0, 3.0).astype(np.float32)
    got = H.binary(ctx, "Pow", ctx.move_tensor(x), ctx.move_tensor(mixed)).get_data()
    assert (got.view(np.uint32) == want.view(np.uint32))[~np.isnan(want) & (mixed == 2.0)].all()
    cubes, fine = ref.binary("Pow", x, mixed), (mixed == 3.0) & np.isfinite(want)
    assert ulp_diff(got[fine], cubes[fine]).max() <= 1  # (a double power is right far beyond fp32: ties only)


def test_sigmoid_over_the_whole_range(ctx):
    x = np.concatenate([np.linspace(-60, 60, 200003), [-12.0, 40.0, np.nextafter(np.float32(-12), np.float32(-13)), 1e30, -1e30,
                                                       np.inf, -np.inf, np.nan, 0.0]]).astype(np.float32)
    got = H.unary(ctx, "Sigmoid", ctx.move_tensor(x)).get_data()
    want = ref.unary("Sigmoid", x)
    assert np.isnan(got[np.isnan(x)]).all()
    # down to -12 the reference's cancelled sum is right to 2^-53 / sigmoid(-12), under 2^-35: only a value that lies
    # that close to a rounding boundary may land one ulp away from it, or from the value itself
    true = 1.0 / (1.0 + np.exp(-x[x >= -12].astype(np.float64)))
    assert ulp_diff(got[x >= -12], true.astype(np.float32)).max() <= 1
    near = x >= -12
    assert ulp_diff(got[near], want[near]).max() <= 1
    # below, both sides form tanh + 1, whose last place is 2^-53 (a double tanh is right to two of them)
    far = x < -12
    assert (np.abs(got[far].astype(np.float64) - want[far]) <= 2.0 ** -51 + 2.0 ** -23 * want[far]).all()


@pytest.mark.parametrize("rows,length", [(1, 65), (5, 256), (4095, 256), (4096, 256), (4097, 255), (5003, 65), (4099, 68), (9001, 257),
                                         (3, 260), (7, 1024), (6, 4099), (2, 100004)])
def test_row_means(ctx, rows, length):
    x = np.random.default_rng(rows + length).standard_normal((rows, length)).astype(np.float32)
    got = H.reduce_mean(ctx, ctx.move_tensor(x), [-1], 0).get_data()
    want = x.astype(np.float64).mean(1)
    slack = length * 2.0 ** -52 * np.abs(x.astype(np.float64)).mean(1)
    assert (np.abs(got - want) <= 2.0 ** -24 * np.abs(want) * 1.0001 + slack).all()


# one pass of a mean over several axes: rows of any length, as few and as many pieces a lane as each form requests ahead
@pytest.mark.parametrize("rows,length", [(4100, 3), (4100, 16), (4100, 18), (4100, 33), (4100, 60), (4100, 64), (10240, 255), (10239, 255), (5, 2), (5, 63),
                                         (5, 65), (5, 129), (5, 257), (9, 513), (9, 512), (9, 1028)])
def test_row_sums_with_another_divisor(ctx, rows, length):
    x = np.random.default_rng(rows + length).standard_normal((rows, length)).astype(np.float32)
    tx, y = ctx.move_tensor(x), ctx.empty_tensor([rows])
    capi.call("wdh_reduce_axis", tx.handle, y.handle, rows, length, 1, 7 * length)
    want = x.astype(np.float64).sum(1) / (7 * length)
    slack = 2.0 ** -52 * np.abs(x.astype(np.float64)).sum(1) / 7
    assert (np.abs(y.get_data() - want) <= 2.0 ** -24 * np.abs(want) * 1.0001 + slack).all()
