"""The scale kernel's strips cut into two and four bands, where the block form
is not taken (a strip width is set): level sizes around the 64-column,
128-column, 8-row and 4-row marks, last bands that are partial or empty, every
plane format and both map forms, against the oracle's form of each.

Tolerance: the pixels and the FP32 block sums are the oracle's, so the norms
differ by the order of the FP64 sums, as in test_gpu_scale_parts.py: 1e-10.
"""
from __future__ import annotations

import os
import subprocess
import tempfile

import numpy as np
import pytest

import vqm_amd
from conftest import ROOT, random_pair
from vqm_amd import DeviceBuffer, Image, ImageFormat, MapForm, Size, Ssimulacra2Batch, Ssimulacra2Config, Ssimulacra2Pipeline

REL = 1e-10
EDGES = [(9, 15), (63, 17), (64, 16), (65, 33), (76, 24), (127, 40), (129, 23), (192, 65), (257, 121)]
# Batches of 200 pairs: size, strip height; four bands each.
FOURS = [((63, 17), 64), ((65, 33), 64), ((76, 24), 64), ((96, 64), 64), ((127, 40), 64), ((257, 121), 128)]
FORMS = [(vqm_amd.PLANES_F32, MapForm.Reference), (vqm_amd.PLANES_F32, MapForm.Difference),
         (vqm_amd.PLANES_F16, MapForm.Reference), (vqm_amd.PLANES_BF16, MapForm.Reference),
         (vqm_amd.PLANES_U16, MapForm.Difference)]


def test_band_counts():
    """The shapes below are what the plans take (host only)."""
    asked, want = [], []
    for planes in range(4):
        for cols in (64, 128):
            for w, h in EDGES:
                asked.append((w, h, planes, cols, 0))
                want.append((16, 2))
        for (w, h), rows in FOURS:
            asked.append((w, h, planes, 128, 200))
            want.append((rows, 4))
    with tempfile.TemporaryDirectory() as tmp:
        exe = os.path.join(tmp, "band_shapes_dump")
        subprocess.run(["g++", "-std=c++20", "-O1", "-Wall",
                        "-I", os.path.join(ROOT, "include"),
                        "-I", os.path.join(ROOT, "vqm_amd", "csrc"),
                        os.path.join(ROOT, "tests", "cpp", "band_shapes_dump.cc"),
                        os.path.join(ROOT, "vqm_amd", "csrc", "ss2_host.cc"),
                        os.path.join(ROOT, "vqm_amd", "csrc", "ss2_source.cc"),
                        "-o", exe], check=True)
        r = subprocess.run([exe], input="\n".join(" ".join(map(str, a)) for a in asked), capture_output=True,
                           text=True, timeout=300, check=True)
    got = [tuple(map(int, line.split())) for line in r.stdout.splitlines()]
    assert dict(zip(asked, got)) == dict(zip(asked, want))


@pytest.mark.gpu
@pytest.mark.parametrize("cols", [64, 128])
@pytest.mark.parametrize("planes,map_form", FORMS)
def test_two_bands(oracle_lib, planes, map_form, cols):
    for i, (w, h) in enumerate(EDGES):
        print(f"two bands {w}x{h} planes {planes} map {int(map_form)} columns {cols}", flush=True)
        a, b = random_pair(w, h, seed=700 + i)
        ia, ib = (Image(Size(w, h), ImageFormat.srgb8(), x) for x in (a, b))
        _, want, _ = oracle_lib.compute(oracle_lib.form_for(planes, int(map_form)), w, h, a, b)
        with Ssimulacra2Pipeline(Ssimulacra2Config(size=Size(w, h), plane_format=planes, map_form=map_form,
                                                   strip_cols=cols)) as p:
            np.testing.assert_allclose(p.Compute(ia, ib).norms(), want, rtol=REL, atol=0)
            assert not p.Compute(ia, ia).norms().any()


@pytest.mark.gpu
@pytest.mark.parametrize("planes,map_form", FORMS)
def test_four_bands(oracle_lib, planes, map_form):
    for i, ((w, h), _) in enumerate(FOURS):
        print(f"four bands {w}x{h} planes {planes} map {int(map_form)}", flush=True)
        a, b = random_pair(w, h, seed=800 + i)
        da, db = DeviceBuffer(a.nbytes), DeviceBuffer(b.nbytes)
        da.upload(a)
        db.upload(b)
        _, want, _ = oracle_lib.compute(oracle_lib.form_for(planes, int(map_form)), w, h, a, b)
        batch = Ssimulacra2Batch(200, plane_format=planes, map_form=int(map_form), strip_cols=128)
        got = batch.Finish(batch.Submit([(da.ptr, db.ptr, w, h)] * 200), raw=True)[1]
        batch.close()
        np.testing.assert_allclose(got[0], want, rtol=REL, atol=0)
        assert (got == got[0]).all()
