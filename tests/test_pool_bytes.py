"""Workspaces of batches and servers against a device-memory budget: a budget
that holds a pair's planes and one partial sum a strip holds the pair, whatever
parts its strips are cut into."""
from __future__ import annotations

import os
import subprocess
import tempfile

import pytest

from conftest import ROOT

# A 1024x1024 pair in FP32 planes, strips of 64 rows, counted with one sum a
# strip (printed by pool_bytes_test.cc).
BYTES_1024 = 14970624


def test_pool_bytes():
    """Builds and runs tests/cpp/pool_bytes_test.cc (host only)."""
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "pool_bytes_test")
        subprocess.run(["g++", "-std=c++20", "-O1", "-Wall",
                        "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "vqm_amd", "csrc"),
                        os.path.join(ROOT, "tests", "cpp", "pool_bytes_test.cc"),
                        os.path.join(ROOT, "vqm_amd", "csrc", "ss2_host.cc"),
                        os.path.join(ROOT, "vqm_amd", "csrc", "ss2_source.cc"),
                        "-o", exe], check=True)
        r = subprocess.run([exe], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stderr
        assert int(r.stdout) == BYTES_1024


@pytest.mark.gpu
@pytest.mark.parametrize("engine", ["batch", "server"])
def test_a_budget_of_one_sum_a_strip_holds_the_pair(engine):
    import numpy as np
    from vqm_amd import DeviceBuffer, Ssimulacra2Batch, Ssimulacra2Server, synth

    a, b = synth.pair(1, 1, 1024, 1024, synth.STRENGTHS[1])
    da, db = DeviceBuffer(a.nbytes), DeviceBuffer(b.nbytes)
    da.upload(a)
    db.upload(b)
    pair = (da.ptr, db.ptr, 1024, 1024)

    def norms(budget):
        if engine == "server":
            with Ssimulacra2Server(lanes=1, strip_rows=64, hbm_budget=budget) as server:
                return np.asarray(server.Wait(server.SubmitDevice(*pair)).norms)
        batch = Ssimulacra2Batch(1, strip_rows=64, hbm_budget=budget)
        try:
            return batch.Finish(batch.Submit([pair]), raw=True)[1][0]
        finally:
            batch.close()

    free = norms(0)
    assert free.any()
    np.testing.assert_array_equal(norms(BYTES_1024), free)
