"""The allocation-free entry point next to the largest pair it takes, where
the partial sums of a strip's parts reach past 128 MiB of scratch: the norms of
a pipeline, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest

import vqm_amd
from test_zz_no_alloc import noalloc, pipeline, upload_pair
from vqm_amd import DeviceBuffer, Size, Ssimulacra2Config
from vqm_amd import _lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h,planes", [(1692, 5271, vqm_amd.PLANES_F32), (6798, 2770, vqm_amd.PLANES_U16)])
def test_noalloc_next_to_its_limit(w, h, planes):
    print(f"noalloc {w}x{h} planes {planes}", flush=True)
    out = DeviceBuffer(108 * 8)
    cfg = Ssimulacra2Config(size=Size(w, h), plane_format=planes)
    da, db = upload_pair(w, h, 4)
    status, scales = noalloc(cfg, da, db, out)
    assert status == 0, L.lib().vqm_last_error()
    assert L.lib().vqm_device_synchronize() == 0
    got = out.download().view(np.float64)
    n, want = pipeline(cfg, da, db)
    assert scales == n
    assert got.any() and np.array_equal(got, want)
    for buffer in (da, db, out):
        buffer.free()
