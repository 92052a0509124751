"""What products and convolutions owe without any tolerance: the sum over nothing."""
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
