"""GPU parity of the PageRank row sums at the sizes where their cut into row
blocks, wave rows and workgroup rows changes: in-degrees around the block,
tile and long-row limits, runs of them, and stretches of empty rows; resident
with both offset widths, and with most rows streamed.  Reference mode must
equal the oracle's sequential FP64 sums bit for bit; normalised mode meets the
L1 bound of 1e-5 against FP64."""
import numpy as np
import pytest

import ascetic_amd as A
from ascetic_amd import _abi
from oracle import oracle as O

pytestmark = pytest.mark.gpu

EDGES = [1, 2, 255, 256, 257, 511, 512, 513, 1023, 1024, 1025, 1535, 1536, 1537, 2047, 2048, 2049, 4095, 4096, 4097]


def in_csr(degrees, seed):
    rng = np.random.default_rng(seed)
    off = np.zeros(len(degrees) + 1, np.uint64)
    off[1:] = np.cumsum(degrees)
    src = rng.integers(0, len(degrees), int(off[-1])).astype(np.uint32)
    return off, src, np.bincount(src, minlength=len(degrees)).astype(np.uint32)


CASES = {
    "limits": EDGES + [0] * 300 + EDGES[::-1] + [3] * 700,
    "runs": [511] * 9 + [512] * 3 + [511] * 600 + [0] * 255 + [1] * 257,
    "long_first": [20000, 9000, 4096] + [0] * 513 + [7] * 1000,
    "long_last": [6] * 1021 + [0] * 3 + [30011],
    "one_vertex": [5],
    "no_edges": [0] * 300,
}


@pytest.mark.parametrize("width", [np.uint32, np.uint64])
@pytest.mark.parametrize("case", sorted(CASES))
def test_rows_resident(gpu_ctx, case, width):
    off, src, od = in_csr(CASES[case], 11)
    csr = O.CSR(off, src)
    ref, rst = O.pr_ref(csr, od)
    norm, res = O.pr_norm(csr, od, 0.85, 20)
    with gpu_ctx.from_arrays(off.astype(width), src, out_degree=od) as g:
        for _ in range(2):   # the second run reuses the plan
            r, _, st = g.pagerank(mode=_abi.PR_REFERENCE)
            assert st["iterations"] == rst["iterations"]
            assert np.array_equal(r, ref)
            r, got, _ = g.pagerank(iterations=20)
            assert np.abs(r.astype(np.float64) - norm).sum() <= 1e-5
            assert np.allclose(got, res, rtol=1e-3, atol=1e-7)


@pytest.mark.parametrize("case", ["limits", "long_first", "long_last"])
def test_rows_streamed(case):
    off, src, od = in_csr(CASES[case], 12)
    csr = O.CSR(off, src)
    ref, _ = O.pr_ref(csr, od)
    norm, _ = O.pr_norm(csr, od, 0.85, 20)
    with A.Context(edge_budget_bytes=4 * (len(src) // 4), part_bytes=4 * 8192) as ctx:
        with ctx.from_arrays(off, src, out_degree=od) as g:
            r, _, _ = g.pagerank(mode=_abi.PR_REFERENCE)
            assert np.array_equal(r, ref)
            r, _, _ = g.pagerank(iterations=20)
            assert np.abs(r.astype(np.float64) - norm).sum() <= 1e-5


def test_reference_mode_iteration_cap(gpu_ctx):
    off, src, od = in_csr(CASES["limits"], 13)
    with gpu_ctx.from_arrays(off, src, out_degree=od) as g:
        r3, _, st = g.pagerank(mode=_abi.PR_REFERENCE, max_iterations=3)
        assert st["iterations"] == 3
        # three power steps from 1/V; no vertex that still moves has stopped
        full, _, _ = g.pagerank(mode=_abi.PR_REFERENCE)
        again, _, _ = g.pagerank(mode=_abi.PR_REFERENCE, max_iterations=3)
    assert np.array_equal(r3, again) and not np.array_equal(r3, full)
