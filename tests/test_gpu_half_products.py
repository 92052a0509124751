"""Products on the f16 matrix cores (operands in two f16 parts, one of them packed) against sums in 64 bits and against the fp32
instruction."""
import numpy as np
import pytest

from webdnn_amd import hostops as H

pytestmark = pytest.mark.gpu

TILES = {2: "128x256", 3: "128x128", 4: "64x128", 5: "64x128"}   # of products: columns are packed


@pytest.fixture
def half(ctx):
    def use(value, chunks=-1):
        ctx.set_option("half_products", value)
        ctx.set_option("split_k", chunks if value > 1 else -1)
    yield use
    use(1)
    ctx.set_option("split_products", 1)


def product(ctx, a, b, transposed, bias=None, r=None, epilogue=None):
    tb = ctx.move_tensor(np.ascontiguousarray(b.T) if transposed else b)
    if r is not None:
        return H.matmul(ctx, ctx.move_tensor(a), tb, ctx.move_tensor(bias), ctx.move_tensor(r), epilogue).get_data()
    return H.gemm(ctx, ctx.move_tensor(a), tb, None if bias is None else ctx.move_tensor(bias), trans_b=int(transposed), epilogue=epilogue).get_data()


def within(got, want, magnitudes, k):
    """Two parts are off by 2^-23 at most and leave out 2^-22 (eight units of 2^-24 with both operands); a chain of at most k
    roundings of half an ulp of the sum of magnitudes."""
    return (np.abs(got - want) <= (k + 16) * 2.0 ** -24 * magnitudes + 1e-37).all()


# less than a block, one, a ragged last one, an odd and an even number; edges of tiles and of strips in both directions
@pytest.mark.parametrize("mode", sorted(TILES))
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("m,n,k,chunks", [(64, 64, 16, 1), (5, 20, 64, 1), (65, 132, 72, 1), (128, 256, 128, 1), (129, 260, 200, 1), (260, 100, 520, 2), (63, 516, 648, 4)])
def test_tiles_and_edges(ctx, half, mode, transposed, m, n, k, chunks):
    rng = np.random.default_rng(m + n + k)
    a, b = rng.standard_normal((m, k)).astype(np.float32), (rng.standard_normal((k, n)) * 0.03).astype(np.float32)
    bias, r = rng.standard_normal(n).astype(np.float32), rng.standard_normal((m, n)).astype(np.float32)
    half(mode, chunks)
    got = product(ctx, a, b, transposed, bias, None if transposed else r, "relu")
    plan = ctx.last_plan()
    assert plan["tile"] == TILES[mode] and plan["split"] == chunks, plan
    a, b = a.astype(np.float64), b.astype(np.float64)
    extra = bias + (0.0 if transposed else r)
    assert within(got, np.maximum(a @ b + extra, 0), np.abs(a) @ np.abs(b) + np.abs(extra), k)


@pytest.mark.parametrize("k", [1024, 4096])
@pytest.mark.parametrize("relu", [False, True])
def test_errors_are_no_larger_than_those_of_bfloat16_parts(ctx, half, k, relu):
    """2-norms against 64 bits, both uncut, and no drift to one side."""
    rng = np.random.default_rng(k)
    a, b = rng.standard_normal((512, k)).astype(np.float32), (rng.standard_normal((k, 512)) * 0.03).astype(np.float32)
    if relu:
        a, b = np.maximum(a, 0), np.abs(b)
    want = a.astype(np.float64) @ b.astype(np.float64)
    err = {}
    ctx.set_option("gemm_wavesplit", 0)
    try:
        half(0)
        ctx.set_option("split_products", 6)
        ctx.set_option("split_k", 1)
        got = product(ctx, a, b, True)
        err["bf16"] = np.linalg.norm(got - want) / np.linalg.norm(want)
        ctx.set_option("split_products", 1)
        half(3, 1)
        got = product(ctx, a, b, True)
        err["f16"] = np.linalg.norm(got - want) / np.linalg.norm(want)
    finally:
        ctx.set_option("gemm_wavesplit", 1)
    assert err["f16"] <= err["bf16"], err
    drift = float(np.sum((got - want) * np.sign(want)) / np.sum(np.abs(want)))
    assert abs(drift) <= 2.0 ** -26, drift


def uniform(rng, shape, exponent):
    return (rng.uniform(1, 2, shape) * 2.0 ** exponent * rng.choice([-1, 1], shape)).astype(np.float32)


@pytest.mark.parametrize("mode", [2, 4, 5])
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("ea,eb", [(0, 0), (-60, 50), (-120, 100), (100, -120), (-130, 20), (-40, -40)])
def test_any_scale(ctx, half, mode, transposed, ea, eb):
    """Powers of two between operands change nothing: both are scaled to f16's range."""
    rng = np.random.default_rng(7)
    a, b = uniform(rng, (130, 200), ea), uniform(rng, (200, 132), eb)
    half(mode, 1)
    got = product(ctx, a, b, transposed)
    assert ctx.last_plan()["tile"] == TILES[mode]
    a, b = a.astype(np.float64), b.astype(np.float64)
    assert (np.abs(got - a @ b) <= 216 * 2.0 ** -24 * (np.abs(a) @ np.abs(b)) + 200 * 2.0 ** -149).all()


@pytest.mark.parametrize("mode", [2, 3, 4, 5])
@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("kind", ["grows", "shrinks", "alone", "rows", "first"])
def test_magnitudes_that_two_parts_cannot_hold(ctx, half, mode, transposed, kind):
    """Elements far above a tile's first block, far below it with partners that lift them, by themselves against zeros, in rows of
    their own; a first block of zeros."""
    rng = np.random.default_rng(8)
    for swap in (False, True):
        a, b = uniform(rng, (140, 320), 0), uniform(rng, (320, 140), 0)
        if kind == "grows":
            a[3, 200], a[100, 319], b[300, 77] = 2.0 ** 30, -(2.0 ** 90), 2.0 ** 20
        elif kind == "shrinks":
            a[:, 100], b[100] = uniform(rng, 140, -60), uniform(rng, 140, 60)
        elif kind == "alone":
            a[:, 64:], b[:64, 20:60] = uniform(rng, (140, 256), -40), 0
        elif kind == "rows":
            a[17], a[80:90] = uniform(rng, 320, -50), uniform(rng, (10, 320), 40)
        else:
            a[:, :64], a[:, 64:] = 0, uniform(rng, (140, 256), -30)
        if swap:
            a, b = np.ascontiguousarray(b.T), np.ascontiguousarray(a.T)
        half(mode, 1)
        got = product(ctx, a, b, transposed)
        assert ctx.last_plan()["tile"] == TILES[mode]
        a, b = a.astype(np.float64), b.astype(np.float64)
        assert within(got, a @ b, np.abs(a) @ np.abs(b), 320), (kind, swap)


@pytest.mark.parametrize("mode", [2, 4, 5])
@pytest.mark.parametrize("transposed", [False, True])
def test_inf_and_nan(ctx, half, mode, transposed):
    rng = np.random.default_rng(11)
    a, b = rng.standard_normal((200, 104)).astype(np.float32), rng.standard_normal((104, 260)).astype(np.float32)
    a[3, 7], a[70, 99], a[130, 0], b[50, 5], b[99, 250] = np.inf, np.nan, -np.inf, np.inf, -np.inf
    a[5, :], b[:, 9], a[199, :], a[199, :2] = 0, 0, 0, 3e38
    a[64] *= np.float32(1e-38)
    a[65] *= np.float32(1e-42)
    out = {}
    for value in (0, mode):
        half(value, 1)
        ctx.set_option("split_products", 0 if value == 0 else 1)
        out[value] = product(ctx, a, b, transposed)
    assert ctx.last_plan()["tile"] == TILES[mode]
    want, got = out[0], out[mode]
    assert (np.isnan(want) == np.isnan(got)).all()
    assert (np.isposinf(want) == np.isposinf(got)).all() and (np.isneginf(want) == np.isneginf(got)).all()
    finite = np.isfinite(want)
    with np.errstate(all="ignore"):
        magnitudes = np.nan_to_num(np.abs(a.astype(np.float64)), posinf=0) @ np.nan_to_num(np.abs(b.astype(np.float64)), posinf=0)
        assert (np.abs(got.astype(np.float64) - want)[finite] <= (112 * 2.0 ** -23 * magnitudes + 2e-45 * 100)[finite]).all()


def test_a_batch_that_shares_its_weight_has_the_bits_of_one_tall_product(ctx, half):
    rng = np.random.default_rng(12)
    x, w = ctx.move_tensor(rng.standard_normal((8, 512, 4096)).astype(np.float32)), ctx.move_tensor((rng.standard_normal((4096, 4096)) * 0.02).astype(np.float32))
    r = ctx.move_tensor(rng.standard_normal((8, 512, 4096)).astype(np.float32))
    plain = H.matmul(ctx, x, w)
    tall = ctx.last_plan()
    want = H.binary(ctx, "Add", plain, r).get_data()
    assert (H.matmul(ctx, x, w, residual=r).get_data() == want).all()
    assert ctx.last_plan() == tall
    half(0)
    assert not (H.matmul(ctx, x, w).get_data() == plain.get_data()).all()   # (it is one for the f16 instruction)
