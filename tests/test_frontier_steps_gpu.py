"""GPU: top-down steps against the oracle where their work is cut differently:
directed BFS just below and above the size whose steps probe bytes instead of
visited bits, frontiers whose vertices a workgroup takes 16 to 256 at a time,
queues filled past a wave's staging, and SSSP runs whose far pile outlasts
several growing bands, with distances past the 16-bit filter among them."""
import numpy as np
import pytest

import ascetic_amd as A
from ascetic_amd import _abi
from oracle import oracle as O
from tests import graphs as G

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [(1 << 18) - 1, 1 << 18, (1 << 18) + 3])
def test_directed_bfs(gpu_ctx, V):
    off, dst, _ = G.random_graph(V, 6 * V, 3, symmetric=False)
    with gpu_ctx.from_arrays(off, dst) as g:
        for src in (0, V - 1):
            assert np.array_equal(g.bfs(src)[0], O.bfs_queue(O.CSR(off, dst), src))


@pytest.mark.parametrize("n", [3073, 32767, 32768, 65537, 300000])
def test_star_of_stars(gpu_ctx, n):
    """A source, n middle vertices, 2 to 40 leaves each that middle vertices share."""
    r = np.random.default_rng(n)
    deg = r.integers(2, 41, n) if n < 100000 else r.integers(2, 5, n)
    V = 1 + n + 50000
    src = np.concatenate([np.zeros(n, np.int64), np.repeat(np.arange(1, n + 1), deg)])
    dst = np.concatenate([np.arange(1, n + 1), r.integers(1 + n, V, int(deg.sum()))])
    off = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=V))]).astype(np.uint64)
    ew = np.stack([dst, r.integers(1, 200, len(dst))], 1).astype(np.uint32)
    csr = O.CSR(off, ew[:, 0].copy(), ew[:, 1].copy())
    with gpu_ctx.from_arrays(off, ew) as g:
        assert np.array_equal(g.bfs(0)[0], O.bfs_queue(csr, 0))
        assert np.array_equal(g.sssp(0)[0], O.dijkstra(csr, 0))


@pytest.mark.parametrize("wmax,delta", [(255, 0), (60000, 0), (255, 3), (1, 0)])
def test_growing_bands(wmax, delta):
    """A skewed graph with a tail of long paths: bands that take little of the
    far pile grow, and values still equal Dijkstra's."""
    h = A.rmat(15, 16, seed=9, weighted=True, wmax=wmax)
    off, ew = h.offsets().copy(), h.edge_words().copy()
    csr = O.CSR(off, ew[:, 0].copy(), ew[:, 1].copy())
    src = int(np.argmax(np.diff(off)))
    with A.Context(sssp_delta=delta) as ctx, ctx.from_arrays(off, ew) as g:
        for _ in range(2):
            assert np.array_equal(g.sssp(src)[0], O.dijkstra(csr, src))
    h.free()


@pytest.mark.parametrize("n", [15, 2049, 32769, 140001])
def test_served_star(gpu_ctx, n):
    """Served lanes through frontiers of n vertices: passes of 16 to 256 (BFS)
    and 64 (SSSP) vertices, from the hub and from three leaves."""
    r = np.random.default_rng(n)
    V = 2 * n + 1
    a = np.concatenate([np.zeros(n, np.int64), np.arange(1, n + 1)])
    b = np.concatenate([np.arange(1, n + 1), n + 1 + r.integers(0, n, n)])
    w = r.integers(1, 100, 2 * n)
    src, dst, wt = np.concatenate([a, b]), np.concatenate([b, a]), np.concatenate([w, w])
    order = np.argsort(src, kind="stable")
    off = np.concatenate([[0], np.cumsum(np.bincount(src, minlength=V))]).astype(np.uint64)
    ew = np.stack([dst[order], wt[order]], 1).astype(np.uint32)
    csr = O.CSR(off, ew[:, 0].copy(), ew[:, 1].copy())
    sources = [0, 1, n, V - 1]
    with gpu_ctx.from_arrays(off, ew) as g, A.Server(g, lanes=16) as srv:
        outs = [(k, s, np.empty(V, np.uint32)) for s in sources for k in (A.Server.BFS, A.Server.SSSP)]
        for t in [srv.submit(k, s, o) for k, s, o in outs]:
            srv.wait(t)
        for k, s, o in outs:
            assert np.array_equal(o, O.bfs_queue(csr, s) if k == A.Server.BFS else O.dijkstra(csr, s)), (k, s)
