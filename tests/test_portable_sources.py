"""The host side of the library is built wherever a GPU is: its sources take what one kind of processor has from the
compiler (vector types, target_clones behind a guard), not from that processor's own headers."""
import glob
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "smat_amd", "csrc")


@pytest.mark.parametrize("source", [os.path.basename(f) for f in sorted(glob.glob(os.path.join(CSRC, "*.cpp")))])
def test_no_header_of_one_processor(source):
    used = subprocess.run(["g++", "-std=c++17", "-M", os.path.join(CSRC, source)], check=True, capture_output=True, text=True).stdout.split()
    assert any(f.endswith(source) for f in used)
    assert [f for f in used if f.endswith("intrin.h") or f.endswith("arm_neon.h")] == []
