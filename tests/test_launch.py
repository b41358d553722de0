"""Builds and runs tests/cpp/launch_test.cc (host only): the launch bookkeeping
of the kernels."""
from __future__ import annotations

import os
import subprocess
import tempfile

from conftest import ROOT


def test_launch():
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "launch_test")
        subprocess.run(["g++", "-std=c++20", "-O1", "-Wall",
                        "-I", os.path.join(ROOT, "vqm_amd", "csrc"),
                        os.path.join(ROOT, "tests", "cpp", "launch_test.cc"),
                        "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr
