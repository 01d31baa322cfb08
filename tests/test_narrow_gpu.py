"""GPU parity where small traversal steps run back to back in one workgroup
and where they change over to the wide kernels and back: long paths and meshes
(thousands of tiny steps), frontiers on both sides of the 3072-vertex and
8192-edge limits, far piles on both sides of 8192 entries, zero-degree
vertices, zero and huge weights, every band setting.  BFS, SSSP and
label-propagation CC bit-exact against the oracle, from several sources on one
graph (the state is reused)."""
import numpy as np
import pytest

import ascetic_amd as A
from ascetic_amd import _abi
from oracle import oracle as O
from tests import graphs as G

pytestmark = pytest.mark.gpu


def mesh(rows, cols, wmax, seed, directed=False):
    at = np.arange(rows * cols).reshape(rows, cols)
    e = np.concatenate([np.stack([at[:, :-1].ravel(), at[:, 1:].ravel()], 1),
                        np.stack([at[:-1].ravel(), at[1:].ravel()], 1)])
    rng = np.random.default_rng(seed)
    e = e[rng.random(len(e)) < 0.93]
    if directed:
        flip = rng.random(len(e)) < 0.3
        e[flip] = e[flip][:, ::-1]
    w = rng.integers(0, wmax + 1, len(e))
    return G.csr_from_edges(rows * cols, e.tolist(), w.tolist(), symmetric=not directed)


def spokes(n_mid, per_mid, tail, wmax, seed):
    """A hub with n_mid neighbours, each with per_mid leaves, and a path of
    `tail` vertices behind the last leaf: the frontier goes 1, n_mid,
    n_mid * per_mid, 1, 1, ..."""
    e = [(0, 1 + i) for i in range(n_mid)]
    nxt = 1 + n_mid
    for i in range(n_mid):
        e += [(1 + i, nxt + j) for j in range(per_mid)]
        nxt += per_mid
    e += [(nxt - 1 + i, nxt + i) for i in range(tail)]
    rng = np.random.default_rng(seed)
    w = rng.integers(1, wmax + 1, len(e))
    return G.csr_from_edges(nxt + tail + 3, e, w.tolist(), symmetric=True)


GRAPHS = {
    "path": lambda: G.csr_from_edges(5000, [(i, i + 1) for i in range(4990)], [(i * 7) % 50 for i in range(4990)],
                                     symmetric=True),
    "mesh": lambda: mesh(60, 83, 255, 1),
    "mesh_wide": lambda: mesh(700, 600, 9, 2),
    "mesh_directed": lambda: mesh(80, 70, 40, 3, directed=True),
    "under_cap": lambda: spokes(1023, 3, 40, 20, 4),       # 3069 leaves
    "over_cap": lambda: spokes(1024, 3, 40, 20, 5),        # 3072
    "past_cap": lambda: spokes(1025, 3, 40, 20, 6),        # 3075
    "edge_limit": lambda: spokes(8192, 1, 30, 20, 7),
    "past_edge_limit": lambda: spokes(8193, 1, 30, 20, 8),
    "big_far": lambda: spokes(90, 100, 30, 5000, 9),       # ~9000 far entries
    "huge_weights": lambda: mesh(40, 45, 0x7FFFFFF0, 10),
}


@pytest.mark.parametrize("width", [np.uint32, np.uint64])
@pytest.mark.parametrize("name", sorted(GRAPHS))
def test_narrow_steps_exact(gpu_ctx, name, width):
    off, dst, w = GRAPHS[name]()
    csr = O.CSR(off, dst, w)
    V = len(off) - 1
    cc = O.cc_minreach(csr)
    with gpu_ctx.from_arrays(off.astype(width), G.wedges(dst, w)) as g:
        for s in (0, V // 2, V - 1, 0):
            d, _ = g.sssp(s)
            assert np.array_equal(d, O.dijkstra(csr, s)), ("sssp", s)
            lv, _ = g.bfs(s)
            assert np.array_equal(lv, O.bfs_queue(csr, s)), ("bfs", s)
        lab, _ = g.cc()
        assert np.array_equal(lab, cc)


@pytest.mark.parametrize("delta", [-1, 1, 7, 100000])
def test_narrow_bands(delta):
    off, dst, w = mesh(50, 50, 60, 11)
    csr = O.CSR(off, dst, w)
    with A.Context(sssp_delta=delta) as ctx, ctx.from_arrays(off, G.wedges(dst, w)) as g:
        for s in (0, 1301):
            assert np.array_equal(g.sssp(s)[0], O.dijkstra(csr, s))


def test_narrow_plain_paths():
    """Top-down BFS and label propagation forced on the unweighted form."""
    off, dst, _ = mesh(90, 64, 5, 12)
    csr = O.CSR(off, dst)
    with A.Context(bfs_direction=_abi.BFS_TOP_DOWN, cc_method=_abi.CC_LABEL_PROP,
                   value_convention=_abi.VALUES_ZERO_BASED) as ctx, ctx.from_arrays(off, dst) as g:
        lv, _ = g.bfs(77)
        ref = O.bfs_queue(csr, 77).astype(np.int64)
        assert np.array_equal(lv, np.where(ref == len(off), 0xFFFFFFFF, ref - 1).astype(np.uint32))
        assert np.array_equal(g.cc()[0], O.cc_minreach(csr))


def test_narrow_long_run_is_cut():
    """More steps than one launch runs (16384)."""
    n = 40000
    off, dst, w = G.csr_from_edges(n, [(i, i + 1) for i in range(n - 1)], [1] * (n - 1), symmetric=True)
    csr = O.CSR(off, dst, w)
    with A.Context() as ctx, ctx.from_arrays(off, G.wedges(dst, w)) as g:
        lv, st = g.bfs(0)
        assert np.array_equal(lv, O.bfs_queue(csr, 0)) and st["iterations"] == n
        assert np.array_equal(g.sssp(n // 3)[0], O.dijkstra(csr, n // 3))
