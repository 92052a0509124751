"""Downloads in pieces."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_downloads_of_many_pieces(ctx):
    """Sizes around the pieces that downloads and uploads travel in, with more pieces than are in flight."""
    for n in (1, (1 << 18) - 1, 1 << 18, (1 << 18) + 1, 5 * (1 << 18) + 3, 9 * (1 << 18)):
        x = np.random.default_rng(n).standard_normal(n).astype(np.float32)
        t = ctx.move_tensor(x)
        assert (t.get_data() == x).all()
        t.set_data(-x)
        assert (t.get_data() == -x).all()


def test_downloads_of_longer_pieces(ctx):
    """From 64 MiB on pieces double, up to 8 MiB: sizes around each step, ragged ones among them."""
    whole = np.arange((520 << 18) + 5, dtype=np.int32)
    for mib in (64, 65, 129, 257, 520):
        n = (mib << 18) + (5 if mib > 64 else 0)
        t = ctx.move_tensor(whole[:n])
        assert (t.get_data() == whole[:n]).all()
        t.dispose()
