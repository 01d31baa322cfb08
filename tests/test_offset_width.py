"""4-byte edge offsets are used on the device only while a kernel's stride past
the last edge cannot wrap 32 bits (a row next to edge 2^32 would never end)."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include <cstdio>
#include "internal.hpp"
int main() {
    const uint64_t top = uint64_t(1) << 32;
    for (uint64_t E : {uint64_t(0), uint64_t(1) << 31, top - 65536, top - 65535, top - 2048, top - 1, top, 2 * top})
        printf("%d %d ", asc::device_offset_bytes(E, 4), asc::device_offset_bytes(E, 8));
}
"""


@pytest.mark.skipif(shutil.which("g++") is None or not os.path.isdir("/opt/rocm/include"), reason="needs g++ and ROCm")
def test_offset_width(tmp_path):
    src, exe = tmp_path / "width.cpp", tmp_path / "width"
    src.write_text(PROGRAM)
    subprocess.run(["g++", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-O1",
                    "-I", os.path.join(ROOT, "ascetic_amd", "csrc"), str(src), "-o", str(exe),
                    "-L", os.path.join(ROOT, "ascetic_amd"), "-l:libascetic.so", "-L/opt/rocm/lib", "-lamdhip64",
                    "-Wl,-rpath," + os.path.join(ROOT, "ascetic_amd"), "-Wl,-rpath,/opt/rocm/lib", "-pthread"],
                   check=True)
    got = subprocess.run([str(exe)], capture_output=True, text=True, check=True).stdout.split()
    assert got == "4 8 4 8 4 8 8 8 8 8 8 8 8 8 8 8".split()
