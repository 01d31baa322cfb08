"""GPU: a BFS without a result array counts the same active vertices as one
with it, whichever kernels took its levels: small steps in one workgroup,
top-down and bottom-up ones."""
import numpy as np
import pytest

import ascetic_amd as A
from ascetic_amd import _abi

pytestmark = pytest.mark.gpu


def path(n):
    """0 - 1 - ... - (n - 1)"""
    i = np.arange(n - 1)
    u, v = np.concatenate([i, i + 1]), np.concatenate([i + 1, i])
    order = np.lexsort((v, u))
    return np.concatenate([[0], np.cumsum(np.bincount(u, minlength=n))]).astype(np.uint64), v[order].astype(np.uint32)


@pytest.mark.parametrize("direction", [_abi.BFS_AUTO, _abi.BFS_TOP_DOWN])
@pytest.mark.parametrize("graph", ["path", "rmat"])
def test_node_sum_without_output(graph, direction):
    if graph == "path":
        off, dst = path(300)
    else:
        h = A.rmat(16, 16, seed=2)
        off, dst = h.offsets().copy(), h.dst().copy()
        h.free()
    src = int(np.argmax(np.diff(off)))
    with A.Context(bfs_direction=direction) as ctx, ctx.from_arrays(off, dst) as g:
        lv, st = g.bfs(src)
        _, none = g.bfs(src, output=False)
    assert st["node_sum"] == (lv != len(off)).sum()
    assert none["node_sum"] == st["node_sum"]
