"""How many chains one triangular-solve launch may hold (host code, no GPU).

Bars: four launches at once, one for each hardware queue, leave half of the
device to the helpers that their chains wait for, whatever its size; a launch
without helpers has no such limit.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include <cstdio>
#include "chain_slabs.hpp"
int main() {
    for (int cus : {1, 8, 32, 64, 80, 128, 256, 304})
        for (int helpers : {0, 1, 2, 3, 4, 7, 16, 60, 124, 1000})
            std::printf("%d %d %d\\n", cus, helpers, elemamd::chain_slabs(helpers, cus));
}
"""


def test_chain_slabs(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "slabs.cpp", tmp_path / "slabs"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-I" + os.path.join(ROOT, "elemental_amd", "csrc"), str(src), "-o", str(exe)],
                   check=True)
    rows = [tuple(map(int, ln.split())) for ln in subprocess.run([str(exe)], check=True, capture_output=True,
                                                                text=True).stdout.splitlines()]
    assert len(rows) == 80
    for cus, helpers, slabs in rows:
        assert slabs >= 1
        if helpers > 0:
            assert slabs == 1 or 4 * slabs <= cus // 2, (cus, helpers, slabs)
        if helpers > 0 and cus >= 64:
            assert slabs >= 8  # ordinary solves keep theirs
