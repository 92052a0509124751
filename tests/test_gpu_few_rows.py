"""Products of a few rows with a transposed weight, against sums in 64 bits."""
import numpy as np
import pytest

from webdnn_amd import capi
from webdnn_amd import hostops as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m", [1, 2, 3, 4, 5])
@pytest.mark.parametrize("n,k", [(2, 128), (3, 131), (7, 1023), (1000, 2048), (4099, 516), (8192, 128), (4096, 130)])
def test_few_rows(ctx, m, n, k):
    rng = np.random.default_rng(m * 100003 + n * 101 + k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), rng.standard_normal((n, k)).astype(np.float32)
    bias = rng.standard_normal(n).astype(np.float32)
    got = H.gemm(ctx, ctx.move_tensor(a), ctx.move_tensor(b), ctx.move_tensor(bias), 0.5, 2.0, 0, 1, epilogue="relu").get_data()
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    want = np.maximum(0.5 * (a64 @ b64.T) + 2.0 * bias, 0.0)
    # a chain of at most k roundings of half an ulp of the sum of magnitudes, then alpha, beta and the bias
    bound = (k + 4) * 2.0 ** -24 * (0.5 * (np.abs(a64) @ np.abs(b64.T)) + 2.0 * np.abs(bias))
    assert got.shape == want.shape and (np.abs(got - want) <= bound).all()


# K long enough for the loop with four steps in flight, with nothing, less than a wavefront and more of it left over;
# by itself (n from about 4096 on) and shared by the wavefronts of a workgroup
@pytest.mark.parametrize("m", [1, 2, 3, 4])
@pytest.mark.parametrize("n,k", [(4099, 1024), (4096, 1028), (4097, 2052), (4096, 2040), (8192, 1000), (1000, 4096), (11, 4100), (1000, 8188), (10, 12292), (4096, 4097)])
def test_few_rows_of_a_long_k(ctx, m, n, k):
    rng = np.random.default_rng(m * 100003 + n * 101 + k)
    a, b = rng.standard_normal((m, k), dtype=np.float32), rng.standard_normal((n, k), dtype=np.float32)
    got = H.gemm(ctx, ctx.move_tensor(a), ctx.move_tensor(b), None, 1.0, 1.0, 0, 1).get_data()
    plan = ctx.last_plan()
    assert plan["tile"] == "%dx2" % m and plan["split"] == (1 if n >= 4096 else 4), plan
    a64, b64 = a.astype(np.float64), b.astype(np.float64)
    bound = (k + 4) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64.T))
    assert (np.abs(got - a64 @ b64.T) <= bound).all()


# more rows than one and a short K: where the matrix cores' form was measured faster it serves
@pytest.mark.parametrize("batch,m,n,k,few", [(1, 1, 3000, 128, True), (1, 4, 3000, 128, False), (1, 3, 3000, 384, False), (1, 4, 910, 256, True),
                                            (1, 4, 911, 256, False), (1, 4, 1000, 257, True), (1, 2, 16384, 191, False), (1, 2, 16384, 192, True), (1, 4, 8192, 512, True),
                                            (1, 4, 8192, 508, False), (1, 4, 8192, 449, False), (1, 4, 8192, 451, True), (4, 4, 577, 192, False), (32, 3, 200, 255, False), (32, 4, 577, 320, True),
                                            (300, 4, 64, 192, False), (300, 2, 64, 128, False), (300, 2, 200, 128, True), (300, 4, 16, 128, True), (256, 4, 16, 128, False), (4096, 1, 2, 128, True)])
def test_which_form_few_rows_take(ctx, batch, m, n, k, few):
    rng = np.random.default_rng(batch + n + k)
    a, b = rng.standard_normal((batch, m, k), dtype=np.float32), rng.standard_normal((batch, n, k), dtype=np.float32)
    ta, tb, y = ctx.move_tensor(a), ctx.move_tensor(b), ctx.empty_tensor([batch, m, n])
    capi.call("wdh_gemm", ta.handle, tb.handle, 0, y.handle, batch, m, n, k, m * k, k, 1, n * k, 1, k, 0, 0, 1.0, 1.0, 0, 0)
    assert (ctx.last_plan()["tile"] == "%dx2" % m) == few, ctx.last_plan()
    a64, b64 = a.astype(np.float64), b.astype(np.float64).transpose(0, 2, 1)
    bound = (k + 4) * 2.0 ** -24 * (np.abs(a64) @ np.abs(b64))
    assert (np.abs(y.get_data() - a64 @ b64) <= bound).all()


def test_few_rows_agree_with_the_other_form_and_keep_inf_and_nan(ctx):
    rng = np.random.default_rng(5)
    a, b = rng.standard_normal((3, 700)).astype(np.float32), rng.standard_normal((37, 700)).astype(np.float32)
    a[1, 3], b[5, 699], b[36, 0] = np.inf, np.nan, -np.inf
    ta, tb = ctx.move_tensor(a), ctx.move_tensor(b)
    got = H.gemm(ctx, ta, tb, None, 1.0, 1.0, 0, 1).get_data()
    ctx.set_option("gemm_wavesplit", 0)
    try:
        other = H.gemm(ctx, ta, tb, None, 1.0, 1.0, 0, 1).get_data()
    finally:
        ctx.set_option("gemm_wavesplit", 1)
    assert (np.isnan(got) == np.isnan(other)).all() and (np.isinf(got) == np.isinf(other)).all()
    fin = np.isfinite(other)
    assert (got[~fin & ~np.isnan(got)] == other[~fin & ~np.isnan(other)]).all()
    np.testing.assert_allclose(got[fin], other[fin], rtol=0, atol=700 * 2.0 ** -23 * 700)
