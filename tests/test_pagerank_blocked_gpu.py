"""GPU: the blocked PageRank layout where it can go wrong: slices of 2^14
sources and bins of 2^13 destinations that end early, runs padded to octs,
empty bins, rows of 4096 edges and more at the ends of a bin and next to each
other, contributions that differ by 2^20 and more, and out-degrees that do
not belong to the edges.

Tolerance: an iteration rounds a rank and its contribution to FP32 once each,
so 20 of them are off by at most 20 * 2 * 2^-24 = 2.4e-6 of a rank; the sums'
fixed point, 4096 half units of 2^-52 of the largest contribution (below 1/2
here) against ranks of 0.15 / 70000 and more, adds 2.2e-7."""
import numpy as np
import pytest

import ascetic_amd as A
from ascetic_amd import _abi
from oracle import oracle as O

pytestmark = pytest.mark.gpu
TOL = 3e-6


def csc(V, src, dst):
    """In-edges of every vertex, and out-degrees."""
    order = np.argsort(dst, kind="stable")
    off = np.concatenate([[0], np.cumsum(np.bincount(dst, minlength=V))]).astype(np.uint64)
    return off, src[order].astype(np.uint32), np.bincount(src, minlength=V).astype(np.uint32)


def uniform(V, E, seed):
    r = np.random.default_rng(seed)
    return r.integers(0, V, E), r.integers(0, V, E)


def rows(V, lengths, seed):
    """Rows of the given in-degrees, vertex -> edges, over random sources, and
    a ring so that every vertex has an out-edge."""
    r = np.random.default_rng(seed)
    dst = np.concatenate([np.full(n, v) for v, n in lengths.items()] + [(np.arange(V) + 1) % V])
    src = np.concatenate([r.integers(0, V, n) for n in lengths.values()] + [np.arange(V)])
    return src, dst


def close(r, ref):
    assert np.all(np.abs(r.astype(np.float64) - ref) <= TOL * ref)


CASES = {
    "one_vertex": lambda: (1, *uniform(1, 3, 0)),
    "below_a_bin": lambda: (8191, *uniform(8191, 50000, 1)),
    "past_a_bin": lambda: (8193, *uniform(8193, 50000, 2)),
    "past_a_slice": lambda: (16385, *uniform(16385, 70001, 3)),
    "sparse": lambda: (100003, *uniform(100003, 1000, 4)),
    "bins_cut_by_edges": lambda: (9000, *uniform(9000, 400000, 5)),
    # 4095 stays in its bin; 4096 and more are bins of their own
    "long_rows": lambda: (20000, *rows(20000, {0: 4096, 1: 5000, 4000: 4095, 8190: 4096, 8191: 4097, 8192: 20001,
                                               16383: 4094, 19999: 6000}, 6)),
    # every other vertex of a few thousand is heavy
    "around": lambda: (30000, *rows(30000, {2 * i: 4096 + i for i in range(40)}, 7)),
    "all_to_one": lambda: (70000, np.arange(1, 70000), np.zeros(69999, np.int64)),
    # vertex 0 hands out 1/69999 of a rank, the others all of theirs
    "one_to_all": lambda: (70000, np.concatenate([np.zeros(69999, np.int64), np.arange(1, 70000)]),
                           np.concatenate([np.arange(1, 70000), np.zeros(69999, np.int64)])),
}


@pytest.mark.parametrize("width", [np.uint32, np.uint64])
@pytest.mark.parametrize("name", CASES)
def test_blocked_layout(gpu_ctx, name, width):
    V, src, dst = CASES[name]()
    off, ids, od = csc(V, np.asarray(src), np.asarray(dst))
    ref, res = O.pr_norm(O.CSR(off, ids), od, 0.85, 20)
    with gpu_ctx.from_arrays(off.astype(width), ids, out_degree=od) as g:
        for _ in range(2):   # the second run reuses the layout
            r, got, _ = g.pagerank(iterations=20, method=_abi.PR_BLOCKED)
            close(r, ref)
            assert np.allclose(got, res, rtol=1e-3, atol=1e-7)


@pytest.mark.parametrize("V,E", [(1 << 17, 1 << 23), ((1 << 20) + 5, 600000), ((1 << 20) + 5, 100000)])
def test_auto_takes_any_graph(gpu_ctx, V, E):
    """The smallest graphs that AUTO blocks, and one too sparse for it."""
    off, ids, od = csc(V, *uniform(V, E, 8))
    ref, _ = O.pr_norm(O.CSR(off, ids), od, 0.85, 20)
    with gpu_ctx.from_arrays(off, ids, out_degree=od) as g:
        close(g.pagerank(iterations=20)[0], ref)


@pytest.mark.parametrize("iterations", [10, 25])
def test_out_degrees_of_other_edges(gpu_ctx, iterations):
    """300 vertices that all point at each other but claim one out-edge: ranks
    grow by 255 an iteration, past FP32 after 17.  AUTO agrees with the pull,
    infinities and NaN included; BLOCKED by name refuses, every time."""
    V, n = (1 << 20) + 5, 300
    a, b = np.divmod(np.arange(n * n), n)
    s2, d2 = uniform(V, 600000, 9)
    s2, d2 = np.maximum(s2, n), np.maximum(d2, n)   # apart from the 300
    off, ids, od = csc(V, np.concatenate([a, s2]), np.concatenate([b, d2]))
    od[:n] = 1
    with gpu_ctx.from_arrays(off, ids, out_degree=od) as g:
        r, _, _ = g.pagerank(iterations=iterations)
        p, _, _ = g.pagerank(iterations=iterations, method=_abi.PR_PULL)
        for _ in range(2):
            with pytest.raises(A.AscError) as e:
                g.pagerank(method=_abi.PR_BLOCKED)
            assert e.value.code == _abi.ERR_FORMAT
    assert np.isfinite(p).all() == (iterations == 10)
    assert np.array_equal(np.isnan(r), np.isnan(p)) and np.array_equal(np.isinf(r), np.isinf(p))
    ok = np.isfinite(p)
    # beside a sum that outgrows the others by 2^80 these lose their digits: absolute there
    assert np.all(np.abs(r[ok] - p[ok]) <= TOL * p[ok] + 2.0 ** -40 * p[ok].max())
