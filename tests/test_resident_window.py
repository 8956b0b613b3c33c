"""Host check of the on-chip solvers' block and halo shapes
(csrc/resident_window.cpp).

tests/resident_window_check.cpp takes the shapes from the library's own
functions and repeats what the kernels keep in LDS and read from it: every
index inside the allocation, every slot's column where it is read, and every
row that a halo loads in a block that the kernel waits for.  Where boxes are
numbered one after another, a halo loads rows that no column of the block
reaches (rows of the last plane of a box lack the entry whose region is loaded).
"""
import os
import shutil
import subprocess

import pytest

REPO = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(REPO, "t-flows-old-compressible_amd", "csrc")


@pytest.fixture(scope="module")
def program():
    cxx = shutil.which("g++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    out = os.path.join(REPO, "_build", "resident_window_check")
    os.makedirs(os.path.dirname(out), exist_ok=True)
    subprocess.run([cxx, "-O2", "-std=c++17", "-I", CSRC, "-o", out,
                    os.path.join(REPO, "tests", "resident_window_check.cpp"),
                    os.path.join(CSRC, "resident_window.cpp")], check=True)
    return out


def test_halo_rows_are_waited_for(program):
    r = subprocess.run([program], capture_output=True, text=True, timeout=120)
    print(r.stdout)
    assert r.returncode == 0 and "ALL OK" in r.stdout, r.stdout + r.stderr
    beyond = {l.split()[1]: int(l.split("beyond=")[1].split()[0]) for l in r.stdout.splitlines() if "beyond=" in l}
    # the patterns that need more than the columns' reach are among the cases
    for name in ("eight_16_cgs", "two_40x40x41_cgs", "three_70x60x25_cgs"):
        assert beyond[name] > 0, name
