"""Whether two column-major blocks share an element (host code, no GPU): every
pair of small blocks against the sets of their addresses."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include <cstdio>
#include <set>
#include "overlap.hpp"
int main() {
    static double mem[4096];
    double* X = mem + 2048;
    long bad = 0, count = 0, yes = 0;
    for (int ldx : {1, 2, 3, 5})
        for (int rx = 0; rx <= ldx; ++rx)
            for (int cx : {0, 1, 2, 4}) {
                std::set<const double*> in;
                for (int j = 0; j < cx; ++j)
                    for (int i = 0; i < rx; ++i) in.insert(X + i + j * ldx);
                for (int ldy : {1, 2, 3, 5, 7})
                    for (int ry = 0; ry <= ldy; ++ry)
                        for (int cy : {0, 1, 3})
                            for (int d = -30; d <= 30; ++d) {
                                bool want = false;
                                for (int j = 0; j < cy; ++j)
                                    for (int i = 0; i < ry; ++i) want |= in.count(X + d + i + j * ldy) > 0;
                                const bool got = elemamd::blocks_overlap(X, ldx, rx, cx, X + d, ldy, ry, cy);
                                bad += got != want;
                                yes += want;
                                ++count;
                            }
            }
    std::printf("%ld %ld %ld\\n", bad, count, yes);
}
"""


def test_against_address_sets(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    if cxx is None:
        pytest.skip("no C++ compiler")
    src, exe = tmp_path / "overlap.cpp", tmp_path / "overlap"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-O1", "-std=c++17", "-I" + os.path.join(ROOT, "elemental_amd", "csrc"), str(src), "-o",
                    str(exe)], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
    bad, count, yes = map(int, out.split())
    assert count > 100000 and yes > 5000 and bad == 0
