"""GPU: which schedule a PageRank call takes does not depend on the calls
before it, and the tuner sweeps a setting only where the schedule reads it."""
import numpy as np
import pytest

from ascetic_amd import _abi

pytestmark = pytest.mark.gpu

V = (1 << 20) + 5


def pairs(n, seed):
    """n vertices with two in-edges each, so that an FP32 sum of a row does not
    depend on the order of its terms (n = 10000: too sparse for the blocked
    layout, which AUTO takes from 34320 edges on at this V)."""
    r = np.random.default_rng(seed)
    deg = np.zeros(V, np.int64)
    deg[r.choice(V, n, replace=False)] = 2
    off = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64)
    src = np.minimum(r.integers(0, V, 2 * n), r.integers(0, V, 2 * n) // 64).astype(np.uint32)   # out-degrees vary
    return off, src, np.bincount(src, minlength=V).astype(np.uint32)


def test_auto_does_not_remember_a_named_schedule(gpu_ctx):
    off, src, od = pairs(10000, 1)
    with gpu_ctx.from_arrays(off, src, out_degree=od) as g:
        first = g.pagerank(iterations=1)[0].copy()
        named = g.pagerank(iterations=1, method=_abi.PR_BLOCKED)[0].copy()
        again = g.pagerank(iterations=1)[0].copy()
        tiled = g.pagerank(iterations=1, method=_abi.PR_TILED)[0].copy()
    assert np.array_equal(first, tiled)            # (one iteration from equal ranks: every sum is the same each time)
    assert not np.array_equal(named, tiled)        # exact sums against sums rounded to FP32
    assert np.array_equal(again, first)


@pytest.mark.parametrize("n,schedule", [(10000, "tiled"), (100000, "blocked")])
def test_tuner_sweeps_what_the_schedule_reads(gpu_ctx, n, schedule):
    off, src, od = pairs(n, 2)
    with gpu_ctx.from_arrays(off, src, out_degree=od) as g:
        t = g.autotune(budget_ms=10000)
    assert t["pr_group"] == 0 and t["score_ms"] <= t["untuned_ms"]
    if schedule == "tiled":
        assert t["pr_tile_src_bits"] in (13, 14, 15, 16, 17, 18)
    else:
        assert t["pr_tile_src_bits"] == 0 and t["score_ms"] == t["untuned_ms"]
