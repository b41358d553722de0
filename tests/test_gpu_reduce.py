"""The reduction's blocks at the counts of parts where a thread's loop starts,
ends or repeats (1, 255, 256, 257, 1,025 parts a range), at images whose
deeper levels are not stored (zeros), and over pairs of a batch.

Tolerance: the parts' FP64 sums are the oracle's up to the order of at most
2^18 non-negative additions, 2^18 * 2^-53 < 3e-11 relative in the worst case;
1e-10 is the suite's bound.
"""
from __future__ import annotations

import numpy as np
import pytest

from conftest import random_pair
from vqm_amd import DeviceBuffer, Image, ImageFormat, Size, Ssimulacra2Batch, Ssimulacra2Config, Ssimulacra2Pipeline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(8, 8), (16, 8), (64, 2040), (64, 2048), (64, 2056), (40, 8200)])
def test_range_lengths(oracle_lib, w, h):
    a, b = random_pair(w, h, seed=w + h)
    _, want, _ = oracle_lib.compute(oracle_lib.form_for(0, 0), w, h, a, b)
    cfg = Ssimulacra2Config(size=Size(w, h), strip_rows=8, strip_cols=64)
    with Ssimulacra2Pipeline(cfg) as p:
        f = ImageFormat.srgb8()
        got = p.Compute(Image(Size(w, h), f, a), Image(Size(w, h), f, b)).norms()
    np.testing.assert_allclose(got, want, rtol=1e-10, atol=0)


def test_pairs_of_a_batch(oracle_lib):
    sizes = [(8, 8), (72, 2056), (33, 17), (64, 2048)]
    hold, items, want = [], [], []
    for i, (w, h) in enumerate(sizes):
        a, b = random_pair(w, h, seed=i)
        da, db = DeviceBuffer(a.nbytes), DeviceBuffer(b.nbytes)
        da.upload(a)
        db.upload(b)
        hold.append((da, db))
        items.append((da.ptr, db.ptr, w, h))
        want.append(oracle_lib.compute(oracle_lib.form_for(0, 0), w, h, a, b)[1])
    batch = Ssimulacra2Batch(len(sizes), strip_rows=8, strip_cols=64)
    got = batch.Finish(batch.Submit(items))
    batch.close()
    for g, w_ in zip(got, want):
        np.testing.assert_allclose(g.norms(), w_, rtol=1e-10, atol=0)
