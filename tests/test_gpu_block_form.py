"""Batches that mix the scale kernel's two forms in one launch: a geometry
first submitted alone in a small launch takes the block form for good, one
first submitted beside another the strip form.

Tolerance against the oracle: the order of at most 2^18 FP64 additions of
non-negative terms, 2^18 * 2^-53 < 3e-11; 1e-10 is the suite's bound. Between
launches of the same plans the sums are the same bit for bit.
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import random_pair
from vqm_amd import DeviceBuffer, Ssimulacra2Batch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("planes", [0, 3])
@pytest.mark.parametrize("chunks", [1, 2])
def test_mixed_forms(oracle_lib, planes, chunks):
    hold = []

    def pair(w, h, seed):
        a, b = random_pair(w, h, seed=seed)
        da, db = DeviceBuffer(a.nbytes), DeviceBuffer(b.nbytes)
        da.upload(a)
        db.upload(b)
        hold.append((da, db))
        want = oracle_lib.compute(oracle_lib.form_for(planes, 0), w, h, a, b)[1]
        return (da.ptr, db.ptr, w, h), want

    blocks = [pair(97, 65, 1), pair(97, 65, 2)]
    strips = [pair(64, 33, 3), pair(200, 40, 4)]
    batch = Ssimulacra2Batch(4, plane_format=planes, chunks=chunks)

    def score(pairs):
        got = batch.Finish(batch.Submit([p for p, _ in pairs]), raw=True)[1]
        for g, (_, want) in zip(got, pairs):
            np.testing.assert_allclose(g, want, rtol=1e-10, atol=0)
        return got

    alone = score(blocks)
    beside = score(strips)
    for order in ([0, 2, 1, 3], [3, 2, 1, 0]):
        every = [(blocks + strips)[i] for i in order]
        expect = np.concatenate([alone, beside])[order]
        assert np.array_equal(score(every), expect)
    batch.close()
