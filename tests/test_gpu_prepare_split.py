"""The prepare kernel's split form (launches of at most 3,584 tiles) against the
oracle at the edges of its rows, columns and levels, and against the other form
at the same sizes: a batch of enough pairs takes that, and its samples, and
with one strip shape its norms, are the same bit for bit.

Tolerance against the oracle: the order of at most 2^18 FP64 additions of
non-negative terms, 3e-11; 1e-10 is the suite's bound.
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import random_pair
from vqm_amd import DeviceBuffer, Ssimulacra2Batch

pytestmark = pytest.mark.gpu

TILE_W, TILE_H, SPLIT_TILES = 64, 32, 14 * 256


@pytest.mark.parametrize("planes,map_form", [(0, 1), (0, 2), (1, 1), (2, 1), (3, 2)])
def test_split_form(oracle_lib, planes, map_form):
    for w, h in [(8, 8), (9, 15), (61, 16), (62, 17), (63, 18), (65, 31), (66, 33), (67, 49), (129, 47)]:
        print(f"split {w}x{h} planes {planes} map {map_form}", flush=True)
        a, b = random_pair(w, h, seed=w * h)
        da, db = DeviceBuffer(a.nbytes), DeviceBuffer(b.nbytes)
        da.upload(a)
        db.upload(b)
        tiles = 2 * (-(-w // TILE_W)) * (-(-h // TILE_H))
        many = SPLIT_TILES // tiles + 1
        got = []
        for pairs in (1, many):
            batch = Ssimulacra2Batch(pairs, plane_format=planes, map_form=map_form, strip_rows=16, strip_cols=64)
            got.append(batch.Finish(batch.Submit([(da.ptr, db.ptr, w, h)] * pairs), raw=True)[1])
            batch.close()
        want = oracle_lib.compute(oracle_lib.form_for(planes, map_form), w, h, a, b)[1]
        np.testing.assert_allclose(got[0][0], want, rtol=1e-10, atol=0)
        assert (got[1] == got[0][0]).all()
