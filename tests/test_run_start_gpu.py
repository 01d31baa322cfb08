"""The start of a run clears every counter that the run publishes at its end,
whatever an earlier one that failed half way left in them.  The library's own
launch_run_init is called on stale memory; the structs are mirrored
from csrc/traverse.hpp, and DevStats' fields are read from there."""
import ctypes as C
import os
import re

import pytest

from ascetic_amd import _abi
from tests.test_zz_no_alloc import DevBuf, _hip

pytestmark = pytest.mark.gpu

CSRC = os.path.join(os.path.dirname(_abi.__file__), "csrc")


class RunInit(C.Structure):
    _fields_ = ([(n, C.c_void_p) for n in ("val", "stamp", "pstamp", "done", "visited", "val16", "seen8")] +
                [("V", C.c_uint64)] +
                [(n, C.c_void_p) for n in ("slots", "piles", "stats", "dcnt", "q0", "pend0")] +
                [(n, C.c_uint32) for n in ("src", "unreached", "n_res0", "n_pend0")])


def words_of(struct):
    """Names of a struct's members; every one of DevStats' is 8 bytes."""
    text = open(os.path.join(CSRC, "traverse.hpp")).read()
    body = re.search(r"struct %s \{(.*?)\n\};" % struct, text, re.S).group(1)
    body = re.sub(r"//[^\n]*", "", body)
    decl = [d.strip() for d in body.split(";") if d.strip()]
    assert all(d.startswith("unsigned long long ") for d in decl)
    return [n.strip() for d in decl for n in d[len("unsigned long long "):].split(",")]


def test_start_clears_the_counters(gpu_ctx):
    names = words_of("DevStats")
    assert {"reached", "degree_sum", "edges_local", "ticks"} <= set(names)
    hip = _hip()
    stats = DevBuf(hip, 2 * len(names) + 16)
    slots, piles = DevBuf(hip, 4 * 8), DevBuf(hip, 8)   # four Slots and the Piles: 32 bytes each
    start = _abi.load()._ZN3asc15launch_run_initERKNS_7RunInitEiP12ihipStream_t
    start.argtypes, start.restype = [C.c_void_p, C.c_int, C.c_void_p], C.c_int
    a = RunInit(V=5, slots=slots.p, piles=piles.p, stats=stats.p, src=0, unreached=6)
    assert start(C.byref(a), 1, None) == 0
    got = stats.get()
    for b in (stats, slots, piles):
        b.free()
    assert (got[:2 * len(names)] == 0).all() and (got[2 * len(names):] == 0xABABABAB).all()
