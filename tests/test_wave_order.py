"""The lanes of a wave (w3d_wave.h), from the sources and their assembly.

Every exchange between the lanes of a wave through LDS is ordered by the
fenced wave_sync() of w3d_wave.h: a bare scheduling barrier orders no memory,
so that a read of another lane's word, or of the same bytes as another type,
would rest on what the compiler happens to do."""
import glob
import os
import subprocess

import pytest

from warp3d_amd.build import ARCH, hipcc

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "warp3d_amd", "csrc")


def test_wave_barriers_are_fenced():
    found = {}
    for f in sorted(glob.glob(os.path.join(CSRC, "*"))):
        n = open(f).read().count("__builtin_amdgcn_wave_barrier")
        if n:
            found[os.path.basename(f)] = n
    assert found == {"w3d_wave.h": 1}, found
    text = open(os.path.join(CSRC, "w3d_wave.h")).read()
    body = text[text.index("void wave_sync()"):]
    body = body[:body.index("}")].split()
    assert [w for w in body if w.startswith("__builtin")] == [
        '__builtin_amdgcn_fence(__ATOMIC_RELEASE,',
        '__builtin_amdgcn_wave_barrier();',
        '__builtin_amdgcn_fence(__ATOMIC_ACQUIRE,']


def test_a_quad_sums_to_the_same_bits(tmp_path):
    """qsum of a product compiles to a product and two additions: contracted,
    fma(a, b, neighbour's a b) rounds its own side once and the neighbour's
    twice, and the lanes of a quad would not agree."""
    try:
        cc = hipcc()
    except RuntimeError:
        pytest.skip("no hipcc")
    src = tmp_path / "q.hip"
    src.write_text('#include "w3d_wave.h"\n'
                   "__global__ void k(const double* a, double* b) {\n"
                   "  const int i = threadIdx.x;\n"
                   "  b[i] = w3d::qsum(a[i] * b[i]);\n}\n")
    out = subprocess.run([cc, f"--offload-arch={ARCH}", "-O3", "-S",
                          "--cuda-device-only", "-I", CSRC, str(src), "-o",
                          "-"], check=True, capture_output=True, text=True)
    ops = [w for w in out.stdout.split() if w.startswith("v_") and "f64" in w]
    assert ops == ["v_mul_f64", "v_add_f64", "v_add_f64"], ops
