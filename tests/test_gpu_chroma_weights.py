"""The staged chroma weights of the filters of more than two taps, in both
forms of the general prepare: a subsampled frame of random chroma scores like
its FP64 upsampling, where the last tile's columns and rows are partial (a row
or column that took another's weights moves the norms far past the tolerance).

Tolerance: 2e-4, the input tests' bound for rounding.
"""
from __future__ import annotations

import numpy as np
import pytest

import format_ref as R
from test_gpu_formats import ROUNDING, max_norm_delta, yuv_format
from vqm_amd import ChromaFilter, ChromaLocation, Size, Ssimulacra2Config, Ssimulacra2Pipeline

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("w,h", [(16, 16), (68, 36), (132, 20), (1044, 1048)])
@pytest.mark.parametrize("flt", [ChromaFilter.Bicubic, ChromaFilter.Lanczos])
@pytest.mark.parametrize("sub_w,sub_h", [(1, 1), (2, 0), (0, 2), (2, 2)])
def test_filtered_chroma(w, h, flt, sub_w, sub_h):
    print(f"{w}x{h} filter {int(flt)} subsampling {sub_w} {sub_h}", flush=True)
    size, location = Size(w, h), ChromaLocation.TopLeft
    rng = np.random.default_rng(w + 10 * sub_w + sub_h)
    shape = (h >> sub_h, w >> sub_w)
    y, x = np.mgrid[0:h, 0:w]
    planes = {0: (0.2 + 0.6 * (x + y) / (w + h)).astype(np.float32).astype(np.float64),
              1: rng.uniform(-0.2, 0.2, shape).astype(np.float32).astype(np.float64),
              2: rng.uniform(-0.2, 0.2, shape).astype(np.float32).astype(np.float64)}
    up = {0: planes[0]} | {c: R.upsample(planes[c], sub_w, sub_h, flt, location, w, h) for c in (1, 2)}
    with Ssimulacra2Pipeline(Ssimulacra2Config(size=size, chroma_filter=int(flt))) as p:
        a = R.pack(yuv_format(sub_w, sub_h, location), size, planes)
        b = R.pack(yuv_format(0, 0, location), size, up)
        delta = max_norm_delta(p.Compute(a, b), p.Compute(b, b))
    assert delta <= ROUNDING, f"{delta:.3e}"
