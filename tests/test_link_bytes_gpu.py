"""What a streamed run says it moved over the link: BFS and CC leave the split
form's weight bytes on the host (4 of 5 bytes a record), SSSP takes whole
records, and a resident run moves nothing."""
import numpy as np
import pytest

import ascetic_amd as A
from ascetic_amd import _abi

pytestmark = pytest.mark.gpu

MODES = {"gather": _abi.STREAM_GATHER, "zerocopy": _abi.STREAM_ZEROCOPY, "hybrid": _abi.STREAM_HYBRID}


@pytest.mark.parametrize("pack,rec", [(2, 5), (1, 4), (0, 8)])
@pytest.mark.parametrize("mode", list(MODES))
def test_link_bytes(mode, pack, rec):
    h = A.rmat(13, 16, seed=4, weighted=True, wmin=1, wmax=255)
    off, ew = h.offsets().copy(), h.edge_words().copy()
    h.free()
    src = int(np.argmax(np.diff(off)))
    with A.Context(edge_budget_bytes=8 * int(off[-1]) // 3, part_bytes=rec * 8192, stream_mode=MODES[mode],
                   stream_pack=pack) as ctx, ctx.from_arrays(off, ew) as g:
        for run, on_link in ((lambda: g.bfs(src), min(rec, 4) if pack else rec), (lambda: g.sssp(src), rec),
                             (g.cc, min(rec, 4) if pack else rec), (lambda: g.sssp(src), rec)):
            _, st = run()
            assert st["streamed_edges"] > 0 and st["link_bytes"] == on_link * st["streamed_edges"]


def test_resident_moves_nothing(gpu_ctx):
    h = A.rmat(10, 8, seed=4, weighted=True)
    with gpu_ctx.adopt(h) as g:
        for st in (g.bfs(0)[1], g.sssp(0)[1], g.cc()[1]):
            assert st["link_bytes"] == 0 and st["streamed_edges"] == 0
