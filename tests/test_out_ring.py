"""The loop that collects results (out_ring.hpp), with a device played by the
test: a helper that stops inside a copy while every queued piece has arrived
is waited for, a late device too, a device that ends without delivering and a
launch that fails are errors; where the system grants no more threads, the
calling one copies alone."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("out_ring") / "check")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-I", os.path.join(HERE, "..", "ascetic_amd", "csrc"),
                    os.path.join(HERE, "out_ring_check.cpp"), "-o", exe, "-pthread"], check=True)
    return exe


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs g++")
@pytest.mark.parametrize("args", [[], ["no-threads"]])
def test_ring_loop(check, args):
    r = subprocess.run([check, *args], capture_output=True, text=True, timeout=60)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr
