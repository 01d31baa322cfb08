"""GPU: the blocked schedule's sums are as close as FP64 ones where
contributions differ by much.

Tolerance: beyond a spread of 2^13 both schedules sum in FP64, below it a sum
is within 2^-26 of the rank, so a rank rounds to the same FP32 value or the
one beside it: 2^-23 of it."""
import numpy as np
import pytest

from ascetic_amd import _abi

pytestmark = pytest.mark.gpu


def clique_beside_hub(V, K, M):
    """Vertices 0..K-1 all point at each other; M leaves and x point at the
    hub, the hub at x; the others are a ring."""
    hub, x, leaf, ring = K, K + 1, K + 2, K + 2 + M
    deg = np.zeros(V, np.int64)
    deg[:K], deg[hub], deg[x], deg[ring:] = K - 1, M + 1, 1, 1
    core = np.tile(np.arange(K, dtype=np.uint32), (K, 1))[~np.eye(K, dtype=bool)]
    src = np.concatenate([core, [x], np.arange(leaf, ring), [hub], np.roll(np.arange(ring, V), 1)]).astype(np.uint32)
    od = np.ones(V, np.uint32)
    od[:K] = K - 1
    return np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64), src, od


@pytest.mark.parametrize("K,M", [(4095, 1 << 18), (3000, 9000), (3000, 5000)])
def test_small_sums_beside_a_large_contribution(gpu_ctx, K, M):
    V = 1 << 19
    off, src, od = clique_beside_hub(V, K, M)
    assert off[-1] == len(src) and len(src) >= 1 << 23
    with gpu_ctx.from_arrays(off, src, out_degree=od) as g:
        b = g.pagerank(iterations=20, method=_abi.PR_BLOCKED)[0].astype(np.float64)
        a = g.pagerank(iterations=20)[0].astype(np.float64)
        p = g.pagerank(iterations=20, method=_abi.PR_PULL)[0].astype(np.float64)
    assert np.all(np.abs(b - p) <= 2.0 ** -23 * p)
    assert np.all(np.abs(a - p) <= 2.0 ** -23 * p)


def test_small_ranks_beside_growing_ones(gpu_ctx):
    """300 vertices that claim one out-edge and have 300 grow by 255 an
    iteration; the others' ranks keep every digit."""
    V, n = (1 << 20) + 5, 300
    r = np.random.default_rng(9)
    a, b = np.divmod(np.arange(n * n), n)
    s = np.concatenate([a, r.integers(n, V, 600000)])
    d = np.concatenate([b, r.integers(n, V, 600000)])
    order = np.argsort(d, kind="stable")
    off = np.concatenate([[0], np.cumsum(np.bincount(d, minlength=V))]).astype(np.uint64)
    od = np.bincount(s, minlength=V).astype(np.uint32)
    od[:n] = 1
    with gpu_ctx.from_arrays(off, s[order].astype(np.uint32), out_degree=od) as g:
        got = g.pagerank(iterations=10)[0].astype(np.float64)
        p = g.pagerank(iterations=10, method=_abi.PR_PULL)[0].astype(np.float64)
    assert p[:n].min() > 2.0 ** 60 * p[n:].max()
    assert np.all(np.abs(got - p) <= 2.0 ** -23 * p)
