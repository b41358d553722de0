"""Builds and runs tests/cpp/noalloc_sizes_test.cc (host only): the sizes the
allocation-free entry point takes do not depend on the parts that a strip is
cut into, and all of them fit its scratch."""
from __future__ import annotations

import os
import subprocess
import tempfile

from conftest import ROOT


def test_noalloc_sizes():
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "noalloc_sizes_test")
        subprocess.run(["g++", "-std=c++20", "-O1", "-Wall",
                        "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "vqm_amd", "csrc"),
                        os.path.join(ROOT, "tests", "cpp", "noalloc_sizes_test.cc"),
                        os.path.join(ROOT, "vqm_amd", "csrc", "ss2_host.cc"),
                        os.path.join(ROOT, "vqm_amd", "csrc", "ss2_source.cc"),
                        "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr
