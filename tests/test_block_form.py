"""Builds and runs tests/cpp/block_form_test.cc (host only): the plans of the
scale kernel's block form tile every stored plane once and stay inside their
buffers."""
from __future__ import annotations

import os
import subprocess
import tempfile

from conftest import ROOT


def test_block_form():
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "block_form_test")
        subprocess.run(["g++", "-std=c++20", "-O1", "-Wall",
                        "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "vqm_amd", "csrc"),
                        os.path.join(ROOT, "tests", "cpp", "block_form_test.cc"),
                        os.path.join(ROOT, "vqm_amd", "csrc", "ss2_host.cc"),
                        os.path.join(ROOT, "vqm_amd", "csrc", "ss2_source.cc"),
                        "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr
