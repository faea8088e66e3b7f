"""Changing a batch plan's launch forms when device memory runs out (host code;
the three runtime calls involved are the test program's own, no GPU).

Bar: a failed change leaves the plan as it was, so that the same change asked
for again is made and not taken for done.
"""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

PROGRAM = """
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include "elemental_amd.h"
static bool fail = false;
static int allocations = 0, live = 0;
extern "C" int hipMalloc(void** p, size_t bytes) {
    if (fail) return 2;  // hipErrorOutOfMemory
    *p = std::malloc(bytes);
    ++allocations, ++live;
    return 0;
}
extern "C" int hipFree(void* p) {
    if (p != nullptr) --live;
    std::free(p);
    return 0;
}
extern "C" int hipMemcpy(void* dst, const void* src, size_t bytes, int) {
    std::memcpy(dst, src, bytes);
    return 0;
}
int main() {
    const int n[3] = {40, 300, 130}, k[3] = {1, 2, 3}, max_n[2] = {128, 1 << 30}, nb[2] = {64, 128};
    const int step[2] = {0, 0}, pers[2] = {0, 4};
    elemamd_batch_plan* plan = nullptr;
    int rc[6];
    rc[0] = elemamd_batch_plan_create(3, n, k, ELEMAMD_BATCH_F64, 2, max_n, nb, &plan);
    const int before = live;
    fail = true;
    rc[1] = elemamd_batch_set_launch(plan, pers);
    fail = false;
    const int kept = live;
    allocations = 0;
    rc[2] = elemamd_batch_set_launch(plan, step);  // the form that it still has
    const int same = allocations;
    rc[3] = elemamd_batch_set_launch(plan, pers);
    const int changed = allocations - same;
    rc[4] = elemamd_batch_set_launch(plan, pers);
    const int again = allocations - same - changed, after = live;
    rc[5] = elemamd_batch_plan_destroy(plan);
    std::printf("%d %d %d %d %d %d  %d %d %d  %d %d %d %d\\n", rc[0], rc[1], rc[2], rc[3], rc[4], rc[5], same, changed,
                again, before, kept, after, live);
}
"""


def test_failed_change_of_launch_forms(tmp_path):
    cxx = shutil.which("g++") or shutil.which("clang++")
    lib = os.path.join(ROOT, "elemental_amd")
    if cxx is None or not os.path.exists(os.path.join(lib, "libelemental_amd.so")):
        pytest.skip("no C++ compiler or no library (__graft_entry__.build() makes it)")
    src, exe = tmp_path / "plan.cpp", tmp_path / "plan"
    src.write_text(PROGRAM)
    subprocess.run([cxx, "-std=c++17", "-I" + os.path.join(ROOT, "include"), str(src), "-o", str(exe), "-rdynamic",
                    "-L" + lib, "-lelemental_amd", "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath," + lib,
                    "-Wl,-rpath,/opt/rocm/lib"], check=True)
    out = subprocess.run([str(exe)], check=True, capture_output=True, text=True, timeout=100).stdout.split()
    created, failed, to_same, to_pers, twice, destroyed, same, changed, again, before, kept, after, left = map(int, out)
    assert created == to_same == to_pers == twice == destroyed == 0 and failed < 0
    assert same == 0 and again == 0  # nothing to change
    assert changed >= 1  # the new form's table was made
    assert before == kept == after and left == 0
