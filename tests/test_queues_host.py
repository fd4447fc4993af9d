"""The order of a batch's tiles, without a GPU: every tile is run once, whichever
workgroup is fast (tests/queues_check.cpp, compiled here with the host compiler
against uvatrmm_amd/csrc/uvt_queues.hpp)."""
import os
import shutil
import subprocess
import tempfile

import pytest

from conftest import ROOT


def test_every_tile_is_run_once():
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    out = os.path.join(tempfile.mkdtemp(), "queues_check")
    subprocess.check_call([cxx, "-std=c++17", "-O2", "-Wall", "-Werror",
                           "-I", os.path.join(ROOT, "uvatrmm_amd", "csrc"),
                           os.path.join(ROOT, "tests", "queues_check.cpp"), "-o", out])
    r = subprocess.run([out], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stderr
    assert r.stdout.strip() == "ok"
