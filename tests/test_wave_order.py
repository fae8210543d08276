"""Every exchange between the lanes of a wave through LDS is ordered by the
fenced wave_sync() of w3d_wave.h: a bare scheduling barrier orders no memory,
so that a read of another lane's word, or of the same bytes as another type,
would rest on what the compiler happens to do."""
import glob
import os

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
    body = text[text.index("void wave_sync()"):].split()
    assert [w for w in body if w.startswith("__builtin")] == [
        '__builtin_amdgcn_fence(__ATOMIC_RELEASE,',
        '__builtin_amdgcn_wave_barrier();',
        '__builtin_amdgcn_fence(__ATOMIC_ACQUIRE,']
