"""GPU: reference PageRank's sums of long rows, which lanes add together, equal
the sequential FP64 sum bit for bit: rows around the limits of a wave's and a
workgroup's tiles, terms that lie halfway between two sums (shares of 2^-k),
terms larger than the sum so far, zeros at the front, and ranks that grow to
infinity because the out-degrees are too small for the edges."""
import numpy as np
import pytest

from ascetic_amd import _abi
from oracle import oracle as O

pytestmark = pytest.mark.gpu

LENGTHS = [512, 513, 575, 1023, 1024, 1025, 4095, 4096, 4097, 6143, 6144, 8191, 8192, 8193, 20001, 70000]


def rows_of(V, lengths, seed):
    """Vertex i has lengths[i] in-edges in random order, the others one each."""
    r = np.random.default_rng(seed)
    deg = np.ones(V, np.int64)
    deg[:len(lengths)] = lengths
    off = np.concatenate([[0], np.cumsum(deg)]).astype(np.uint64)
    return off, r.integers(0, V, int(off[-1])).astype(np.uint32)


def with_dangling(off, ids, od, iterations):
    """The oracle's iteration, but a vertex without out-edges hands out 0 (the
    oracle divides by its out-degree): the longer rows by cumsum, which adds
    one after the other."""
    V = len(off) - 1
    val, active = np.full(V, 1.0 / V), np.ones(V, bool)
    for it in range(iterations):
        c = np.where(od > 0, val / np.maximum(od, 1), 0.0)[ids]
        s = c[off[:-1].astype(np.int64)]
        for v in np.flatnonzero(np.diff(off) > 1):
            s[v] = np.cumsum(c[int(off[v]):int(off[v + 1])])[-1]
        t = 0.15 + 0.85 * s
        active &= np.abs(t - val) > 0.001
        val = np.where(active, t, val)
        if not active.any():
            break
    return val, {"iterations": it + 1}


def same(gpu_ctx, off, ids, od, iterations):
    ref, st = (O.pr_ref(O.CSR(off, ids), od, max_iter=iterations) if od.all()
               else with_dangling(off, ids, od, iterations))
    with gpu_ctx.from_arrays(off, ids, out_degree=od) as g:
        r, _, got = g.pagerank(mode=_abi.PR_REFERENCE, max_iterations=iterations)
    assert got["iterations"] == st["iterations"]
    assert np.array_equal(r, ref, equal_nan=True)


@pytest.mark.parametrize("shares", ["degrees", "powers", "equal", "spread", "none_at_first"])
def test_ordered_rows(gpu_ctx, shares):
    V = 30000
    off, ids = rows_of(V, LENGTHS, 3)
    r = np.random.default_rng(4)
    od = {
        "degrees": lambda: np.bincount(ids, minlength=V),
        "powers": lambda: 1 << r.integers(0, 31, V),          # halfway terms at every size of the sum
        "equal": lambda: np.full(V, 8),
        "spread": lambda: np.where(r.random(V) < 1e-3, 1, 2 ** 31),
        "none_at_first": lambda: np.where(np.arange(V) < V // 2, 0, 3),
    }[shares]().astype(np.uint32)
    if shares == "none_at_first":   # rows in ascending order start with vertices that hand out nothing
        for v in range(len(LENGTHS)):
            ids[off[v]:off[v + 1]].sort()
    same(gpu_ctx, off, ids, od, 12)


def test_ordered_rows_to_infinity(gpu_ctx):
    """600 vertices that all point at each other and claim one out-edge: x 510
    an iteration, past FP64 after 114."""
    n = 600
    off = (np.arange(n + 1) * n).astype(np.uint64)
    ids = np.tile(np.arange(n, dtype=np.uint32), n)
    same(gpu_ctx, off, ids, np.ones(n, np.uint32), 118)
