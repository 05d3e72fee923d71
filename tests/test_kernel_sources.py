"""Rules of the kernels' sources that no run shows: what a compiler's schedule happens to hold is not relied on."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "sglang_security_amd", "csrc")


def test_ring_barriers_wait_for_lds_reads():
    """A barrier that frees an LDS stage for the next direct load follows a counted wait for the loads under way; the same
    wait covers the wave's reads of the stage it gives up."""
    seen = 0
    for path in glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip")):
        src = open(path).read()
        for m in re.finditer(r'asm volatile\("s_waitcnt ([^"]*)" ::"n"[^;]*;\s*__builtin_amdgcn_s_barrier\(\)', src):
            seen += 1
            assert "vmcnt" in m[1] and "lgkmcnt(0)" in m[1], (os.path.basename(path), m[0])
    assert seen >= 2


def test_matrix_instructions_are_the_compilers():
    """A matrix instruction written out as text leaves its sums some cycles later without the compiler knowing: it may place a copy of them
    right behind.  Only the builtins carry that."""
    for path in glob.glob(os.path.join(CSRC, "*.h")) + glob.glob(os.path.join(CSRC, "*.hip")):
        src = re.sub(r"//[^\n]*", "", open(path).read())
        assert not re.search(r'"[^"]*v_s?mfma', src), os.path.basename(path)
