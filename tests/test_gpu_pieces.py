"""Gather of whole runs, MaxPool bands and broadcasts in pieces of one, two and four elements."""
import numpy as np
import pytest

from oracle import ref
from webdnn_amd import capi
from webdnn_amd import hostops as H

pytestmark = pytest.mark.gpu


# runs of less than, exactly and more than a wavefront's least, in pieces of one, two and four; of one and several chunks, the last ragged
@pytest.mark.parametrize("inner", [47, 48, 49, 96, 98, 191, 192, 196, 1023, 1024, 1025, 2050, 4096, 4100, 9998])
@pytest.mark.parametrize("outer,axis,n", [(1, 5, 7), (3, 4, 1), (6, 1, 3)])
def test_gather_of_runs(ctx, inner, outer, axis, n):
    rng = np.random.default_rng(inner + outer)
    x = rng.standard_normal((outer, axis, inner)).astype(np.float32)
    idx = rng.integers(-axis, axis, n).astype(np.int32)
    y = H.gather(ctx, ctx.move_tensor(x), ctx.move_tensor(idx), 1).get_data()
    assert (y == x[:, idx]).all()
    xi = rng.integers(-9, 9, x.shape).astype(np.int32)
    assert (H.gather(ctx, ctx.move_tensor(xi), ctx.move_tensor(idx), 1).get_data() == xi[:, idx]).all()


# (a little under and at the limit; 3.2 GB of results)
@pytest.mark.parametrize("runs", [(1 << 24) - 1, 1 << 24])
def test_gather_of_more_runs_than_a_launch_has_workgroups(ctx, runs):
    """2^24 workgroups of 256 threads are one too many for a launch."""
    inner = 49
    x = np.arange(3 * inner, dtype=np.float32).reshape(3, inner)
    idx = (np.arange(runs) % 3).astype(np.int32)
    y = H.gather(ctx, ctx.move_tensor(x), ctx.move_tensor(idx), 0)
    part = np.empty((1000, inner), np.float32)
    for first in (0, runs // 2, runs - 1000):
        capi.call("wdh_read", y.handle, first * inner * 4, part.ctypes.data, part.nbytes)
        assert (part == x[idx[first:first + 1000]]).all()
    y.dispose()
    capi.call("wdh_trim", 0)


def test_gather_out_of_range_reads_the_first_run(ctx):
    x = np.arange(3 * 100, dtype=np.float32).reshape(3, 100)
    idx = np.array([3, -4, 2, 1 << 30], np.int32)
    y = H.gather(ctx, ctx.move_tensor(x), ctx.move_tensor(idx), 0).get_data()
    assert (y == x[[0, 0, 2, 0]]).all()


@pytest.mark.parametrize("w", [64, 62, 63, 126, 200])
@pytest.mark.parametrize("h,kernel,stride,pad", [(40, 3, 2, 1), (33, 2, 2, 0), (50, 5, 3, 2)])
def test_maxpool_bands(ctx, w, h, kernel, stride, pad):
    rng = np.random.default_rng(w + h)
    x = rng.standard_normal((2, 3, h, w)).astype(np.float32)
    x[0, 1, 5, 7] = np.nan
    got = H.maxpool(ctx, ctx.move_tensor(x), [kernel] * 2, pads=[pad] * 4, strides=[stride] * 2).get_data()
    assert (got == ref.maxpool(x, [kernel] * 2, pads=[pad] * 4, strides=[stride] * 2)).all()


# rows of 2 (mod 4) elements: pieces of two, tiles and flat runs; an operand by channel, by column and a scalar
@pytest.mark.parametrize("op", ["Add", "Sub", "Mul", "Div", "Pow"])
@pytest.mark.parametrize("shape,other", [((2, 3, 5, 126), (3, 1, 1)), ((4, 6, 50), (50,)), ((7, 5, 30), (7, 1, 30)), ((3, 1026), (1,)), ((2, 3, 9, 14), (2, 1, 9, 1)),
                                         ((5, 3, 2), (3, 1)), ((4, 130), (4, 1))])
def test_broadcast_in_pieces_of_two(ctx, op, shape, other):
    rng = np.random.default_rng(sum(shape))
    a, b = rng.uniform(0.5, 2, shape).astype(np.float32), rng.uniform(0.5, 2, other).astype(np.float32)
    for l, r in ((a, b), (b, a)):
        got = H.binary(ctx, op, ctx.move_tensor(l), ctx.move_tensor(r)).get_data()
        want = ref.binary(op, l, r)
        if op == "Pow":
            assert np.allclose(got, want, rtol=2e-7, atol=0)
        else:
            assert (got == want).all()
