"""The autotuner's candidates hold the shape that a launch takes untuned."""
from __future__ import annotations

import os
import subprocess
import tempfile

import pytest

from conftest import ROOT, random_pair


def test_tune_shapes():
    """Builds and runs tests/cpp/tune_shapes_test.cc (host only)."""
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "tune_shapes_test")
        subprocess.run(["g++", "-std=c++20", "-O1", "-Wall",
                        "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "vqm_amd", "csrc"),
                        os.path.join(ROOT, "tests", "cpp", "tune_shapes_test.cc"),
                        os.path.join(ROOT, "vqm_amd", "csrc", "ss2_host.cc"),
                        os.path.join(ROOT, "vqm_amd", "csrc", "ss2_source.cc"),
                        "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr


@pytest.mark.gpu
@pytest.mark.parametrize("persistent", [False, True])
def test_tuned_small_launch(oracle_lib, persistent):
    """A tuned launch whose candidates hold the block form (not taken where it
    is persistent) against the oracle, 1e-10 relative: the order of at most
    2^18 FP64 additions of non-negative terms, 2^18 * 2^-53 < 3e-11."""
    import numpy as np
    from vqm_amd import DeviceBuffer, Ssimulacra2Batch

    w, h = 97, 65
    a, b = random_pair(w, h, seed=9)
    da, db = DeviceBuffer(a.nbytes), DeviceBuffer(b.nbytes)
    da.upload(a)
    db.upload(b)
    want = oracle_lib.compute(oracle_lib.form_for(0, 0), w, h, a, b)[1]
    batch = Ssimulacra2Batch(2, autotune=True, persistent=persistent)
    for _ in range(2):
        for got in batch.Finish(batch.Submit([(da.ptr, db.ptr, w, h)] * 2), raw=True)[1]:
            np.testing.assert_allclose(got, want, rtol=1e-10, atol=0)
    batch.close()
