"""Reductions over an inner axis on the GPU, against sums in 64 bits."""
import numpy as np
import pytest

from webdnn_amd import hostops as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,axis", [((3, 31, 5), 1), ((2, 32, 7), 1), ((2, 500, 17), 1), ((1, 33, 16), 1), ((40, 129, 500), 1),
                                        ((300, 63, 255), 1), ((4, 5, 70000), 1), ((1, 71, 66000), 1)])
def test_mean_over_an_inner_axis(ctx, shape, axis):
    x = np.random.default_rng(sum(shape)).standard_normal(shape).astype(np.float32)
    got = H.reduce_mean(ctx, ctx.move_tensor(x), [axis], 0).get_data()
    want = x.astype(np.float64).sum(axis) / shape[axis]
    # sums in double whatever their order: one rounding to fp32, and a sum's double error under cancellation
    slack = shape[axis] * 2.0 ** -52 * np.abs(x.astype(np.float64)).mean(axis)
    assert (np.abs(got - want) <= 2.0 ** -24 * np.abs(want) * 1.0001 + slack).all()
