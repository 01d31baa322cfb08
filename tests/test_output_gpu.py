"""Results on their way to the caller: sizes around the pieces they are sent in
(32768 values; 8 pieces a launch, 16 in flight), every entry point that returns
V values, both value conventions, the reached count and degree sum that are
counted on the way, and served queries of one batch sent together."""
import numpy as np
import pytest

import ascetic_amd as A
from ascetic_amd import _abi

pytestmark = pytest.mark.gpu

P = 32768
SIZES = [1, 2, 3, 1000, P - 1, P, P + 1, 2 * P + 3, 3 * P, 8 * P - 5, 8 * P + 1, 16 * P, 16 * P + 1, 33 * P + 77]


def fan(V):
    """0 -> every odd vertex, every odd vertex -> 0, the even ones alone."""
    odd = np.arange(1, V, 2, dtype=np.uint32)
    off = np.zeros(V + 1, np.uint64)
    deg = np.zeros(V, np.int64)
    deg[0], deg[odd] = len(odd), 1
    off[1:] = np.cumsum(deg)
    return off, np.concatenate([odd, np.zeros(len(odd), np.uint32)])


@pytest.mark.parametrize("zero_based", [False, True])
@pytest.mark.parametrize("V", SIZES)
def test_values_and_counts(V, zero_based):
    off, dst = fan(V)
    edges = np.stack([dst, dst % 5 + 1], axis=1).astype(np.uint32)
    unreached = 0xFFFFFFFF if zero_based else V + 1
    base = 0 if zero_based else 1
    want = np.full(V, unreached, np.uint32)
    odd = np.arange(1, V, 2)
    want[0], want[odd] = base, base + 1
    dist = want.copy()
    # the reference's values never go past V + 1
    d = 1 + odd % 5 + 1
    dist[odd] = np.where(d < V + 1, d - (1 - base), unreached)
    with A.Context(value_convention=_abi.VALUES_ZERO_BASED if zero_based else _abi.VALUES_REFERENCE) as ctx:
        with ctx.from_arrays(off, edges) as g:
            for _ in range(2):
                lv, st = g.bfs(0)
                assert np.array_equal(lv, want)
                assert st["reached"] == 1 + len(odd) and st["reached_degree_sum"] == len(dst)
                dd, st = g.sssp(0)
                assert np.array_equal(dd, dist)
                assert st["reached"] == (dist != unreached).sum()
                lab, st = g.cc()
                cc = np.arange(V, dtype=np.uint32)
                cc[odd] = 0
                assert np.array_equal(lab, cc) and st["reached"] == V and st["reached_degree_sum"] == len(dst)


@pytest.mark.parametrize("V", [1, P - 1, P + 1, 8 * P + 1, 16 * P + 1])
def test_ranks(gpu_ctx, V):
    off, src = fan(V)   # its own transpose
    od = np.diff(off).astype(np.uint32)
    with gpu_ctx.from_arrays(off, src, out_degree=od) as g:
        r, _, _ = g.pagerank(iterations=1)
        r64, _, _ = g.pagerank(mode=_abi.PR_REFERENCE, max_iterations=1, threshold=0.0)
    c = np.where(od > 0, 1.0 / V / np.maximum(od, 1), 0.0)
    s = np.zeros(V)
    odd = np.arange(1, V, 2)
    # the reference mode adds in CSR order: cumsum does too (numpy's sum adds in pairs)
    s[0], s[odd] = np.cumsum(c[odd])[-1] if len(odd) else 0.0, c[0]
    dangling = (od == 0).sum() / V
    assert np.allclose(r, 0.15 / V + 0.85 * (s + dangling / V), rtol=1e-6, atol=0)
    assert np.allclose(r64, 0.15 + 0.85 * s, rtol=1e-12, atol=0)


@pytest.mark.parametrize("V", [3, P + 1, 8 * P + 5])
def test_served_batch(gpu_ctx, V):
    off, dst = fan(V)
    edges = np.stack([dst, np.ones(len(dst))], axis=1).astype(np.uint32)
    rng = np.random.default_rng(V)
    srcs = rng.integers(0, V, 70)
    with gpu_ctx.from_arrays(off, edges) as g, A.Server(g, lanes=64) as srv:
        outs = [np.empty(V, np.uint32) for _ in srcs]
        kinds = [A.Server.BFS if i % 3 else A.Server.SSSP for i in range(len(srcs))]
        for t in [srv.submit(k, int(s), o) for k, s, o in zip(kinds, srcs, outs)]:
            srv.wait(t)
    for s, o in zip(srcs, outs):
        want = np.full(V, V + 1, np.uint32)
        if s % 2 == 0 and s > 0:
            want[s] = 1
        else:
            want[1::2], want[0] = (2, 1) if s == 0 else (3, 2)
            want[s] = 1
        assert np.array_equal(o, np.minimum(want, V + 1)), s
