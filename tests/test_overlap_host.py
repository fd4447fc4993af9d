"""Whether two blocks share an element, without a GPU (tests/overlap_check.cpp,
compiled here with the host compiler against uvatrmm_amd/csrc/uvt_overlap.hpp)."""
import os
import shutil
import subprocess
import tempfile

import pytest

from conftest import ROOT


def test_overlap_of_blocks():
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    out = os.path.join(tempfile.mkdtemp(), "overlap_check")
    subprocess.check_call([cxx, "-std=c++17", "-O2", "-Wall", "-Werror",
                           "-I", os.path.join(ROOT, "uvatrmm_amd", "csrc"),
                           os.path.join(ROOT, "tests", "overlap_check.cpp"), "-o", out])
    r = subprocess.run([out], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip() == "ok"
