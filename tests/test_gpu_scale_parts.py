"""The scale kernel's parts (64 columns by a band of a strip, four source rows
a step) where their edges fall: level widths and heights around the 64-column,
128-column, 8-row and 4-row marks, strips cut into bands, and every plane
format, bit-level with the oracle's form of each configuration.

Tolerance: the kernel's pixels and FP32 block sums are the oracle's, so the
norms differ by the order of at most 2^22 FP64 additions of non-negative
terms: 2^22 * 2^-53 < 1e-9 relative in the worst case and about its square
root, 1e-12, for rounding errors of either sign; 1e-10 is the suite's bound.
"""
from __future__ import annotations

import numpy as np
import pytest

import vqm_amd
from conftest import random_pair
from vqm_amd import Image, ImageFormat, MapForm, Size, Ssimulacra2Config, Ssimulacra2Pipeline

pytestmark = pytest.mark.gpu

REL = 1e-10
EDGES = [(8, 8), (9, 15), (63, 17), (64, 16), (65, 33), (76, 24), (127, 40), (129, 23), (192, 65), (257, 121)]


def norms(w, h, a, b, **cfg):
    with Ssimulacra2Pipeline(Ssimulacra2Config(size=Size(w, h), **cfg)) as p:
        return p.Compute(Image(Size(w, h), ImageFormat.srgb8(), a), Image(Size(w, h), ImageFormat.srgb8(), b)).norms()


@pytest.mark.parametrize("shape", [(0, 0), (8, 64), (24, 128), (104, 64)])
@pytest.mark.parametrize("planes,map_form", [(vqm_amd.PLANES_F32, MapForm.Reference),
                                             (vqm_amd.PLANES_F32, MapForm.Difference),
                                             (vqm_amd.PLANES_F16, MapForm.Reference),
                                             (vqm_amd.PLANES_BF16, MapForm.Reference),
                                             (vqm_amd.PLANES_U16, MapForm.Difference)])
def test_parts_at_their_edges(oracle_lib, planes, map_form, shape):
    """The default shape (bands of a strip) and explicit ones; identical
    images score exactly 100 wherever the parts end."""
    for i, (w, h) in enumerate(EDGES):
        print(f"parts {w}x{h} planes {planes} map {int(map_form)} shape {shape}", flush=True)
        a, b = random_pair(w, h, seed=300 + i)
        cfg = dict(plane_format=planes, map_form=map_form, strip_rows=shape[0], strip_cols=shape[1])
        _, want, _ = oracle_lib.compute(oracle_lib.form_for(planes, int(map_form)), w, h, a, b)
        np.testing.assert_allclose(norms(w, h, a, b, **cfg), want, rtol=REL, atol=0)
        assert not norms(w, h, a, a, **cfg).any()


def test_bands_change_only_the_order_of_the_sums():
    """Sizes whose default strips are cut into two or four bands against
    uncut strips of the same height."""
    for w, h in ((96, 64), (512, 512), (853, 479), (3840, 2160)):
        a, b = random_pair(w, h, seed=w)
        auto = norms(w, h, a, b)
        for rows in (8, 16, 64):
            np.testing.assert_allclose(norms(w, h, a, b, strip_rows=rows), auto, rtol=1e-12, atol=0)
