"""Attention whose queries and keys pass through LDS a few rows at a time: edges of the blocks of 32 rows and keys, of the
wavefronts' shares (one, two and four blocks) and of the head dimension.

The chain of nodes: src/descriptor_runner/operators/cpu/operators/standard/matmul.ts:11-111, softmax.ts:34-57.
"""
import numpy as np
import pytest

from webdnn_amd import hostops as H

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tq,tk", [(1, 1), (31, 33), (33, 256), (32, 257), (65, 511), (5, 513), (34, 993), (3, 1024)])
@pytest.mark.parametrize("heads,d", [(3, 32), (2, 64), (2, 128)])
def test_edges_against_64_bits(ctx, tq, tk, heads, d):
    """Rows of `more` further keys behind the last are NaN and Inf: nothing of them may be seen."""
    rng = np.random.default_rng(tk * d + tq)
    more, w = 5, heads * d
    q = rng.standard_normal((tq, w)).astype(np.float32)
    k, v = (rng.standard_normal((tk + more, w)).astype(np.float32) for _ in range(2))
    k[tk:] = np.nan
    v[tk:] = np.inf
    alpha = np.float32(d ** -0.5)
    y = ctx.empty_tensor([tq, w])
    handles = [ctx.move_tensor(a).handle for a in (q, k, v)]
    H.call("wdh_attention", *handles, y.handle, heads, tq, tk, d, d, w, d, w, d, w, d, w, float(alpha))
    q64, k64, v64 = (a.astype(np.float64).reshape(-1, heads, d) for a in (q, k[:tk], v[:tk]))
    s = np.matmul(q64.transpose(1, 0, 2), k64.transpose(1, 2, 0)) * float(alpha)
    size = np.matmul(np.abs(q64).transpose(1, 0, 2), np.abs(k64).transpose(1, 2, 0)) * float(alpha)
    e = np.exp(s - s.max(-1, keepdims=True))
    want = np.matmul(e / e.sum(-1, keepdims=True), v64.transpose(1, 0, 2)).transpose(1, 0, 2).reshape(tq, w)
    # A score is off by (d/2 + 2) roundings of at most the sum of its terms' sizes, e^x by that and 4 more, its sum by a chain
    # of log2 steps of 64 lanes and 16 pieces (22), the second product by a chain of tk/2 + 16 sums of weights that add up to 1.
    eps = 2.0 ** -24
    bound = (2 * (d / 2 + 2) * size.max() + 4 + 22 + tk / 2 + 16) * eps * np.abs(v64).max()
    assert np.abs(y.get_data().reshape(tq, w) - want).max() <= bound
