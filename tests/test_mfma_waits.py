"""Inline FP64 MFMA statements carry the wait states after which any
instruction may read their result.

The bar is what hipcc itself puts between the builtin and a vector read of its
result; a statement needs as many, because the compiler does not know that it
holds an MFMA and may copy the accumulator right behind it.
"""
import glob
import os
import re
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

PROBE = """
#include <hip/hip_runtime.h>
typedef double d4_t __attribute__((ext_vector_type(4)));
extern "C" __global__ void probe(const double* a, double* out) {
    d4_t c = {a[0], a[1], a[2], a[3]};
    c = __builtin_amdgcn_mfma_f64_16x16x4f64(a[threadIdx.x], a[64 + threadIdx.x], c, 0, 0, 0);
    out[threadIdx.x] = ((c[0] + c[1]) + c[2]) + c[3];
}
"""


def states(line):
    m = re.match(r"s_nop (\d+)", line)
    return int(m.group(1)) + 1 if m else 1


@pytest.fixture(scope="module")
def needed(tmp_path_factory):
    if not os.path.exists(HIPCC):
        pytest.skip("no hipcc")
    d = tmp_path_factory.mktemp("mfma")
    src, out = d / "probe.hip", d / "probe.s"
    src.write_text(PROBE)
    subprocess.run([HIPCC, "-O3", "--offload-arch=gfx950", "--offload-device-only", "-S", str(src), "-o", str(out)],
                   check=True, capture_output=True)
    lines = [ln.split(";")[0].strip() for ln in out.read_text().splitlines()]
    lines = [ln for ln in lines if ln and not ln.startswith(".")]
    at = next(i for i, ln in enumerate(lines) if ln.startswith("v_mfma_f64"))
    n = 0
    for ln in lines[at + 1:]:
        if ln.startswith("v_"):  # the first vector instruction reads the result
            break
        n += states(ln)
    assert 8 <= n <= 64
    return n


def statements():
    for path in sorted(glob.glob(os.path.join(ROOT, "elemental_amd", "csrc", "*"))):
        if not path.endswith((".hip", ".hpp", ".cpp")):
            continue
        for m in re.finditer(r"asm volatile\(((?:\s*\"(?:[^\"\\]|\\.)*\")+)", open(path).read()):
            text = "".join(re.findall(r"\"((?:[^\"\\]|\\.)*)\"", m.group(1)))
            lines = [ln.strip() for ln in text.replace("\\t", " ").split("\\n")]
            if any(ln.startswith("v_mfma_f64") for ln in lines):
                yield os.path.basename(path), lines


def test_wait_states(needed):
    found = list(statements())
    assert found
    for name, lines in found:
        last = max(i for i, ln in enumerate(lines) if ln.startswith("v_mfma_f64"))
        assert sum(states(ln) for ln in lines[last + 1:]) >= needed, name
