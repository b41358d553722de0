"""SMPTE ST 2084 samples far past the curve's range, whose quotient leaves the
fast division's domain and takes the IEEE one, beside ordinary samples of the
same lanes: linear light there is infinite whatever the sample (a denominator
of 1.2e-38, a quotient above 1e36 and its 6.28th power), so that any two such
samples give the same norms bit for bit; ordinary ones do not.
"""
from __future__ import annotations

import numpy as np
import pytest

from vqm_amd import (ColorFamily, ColorPrimaries, Image, ImageFormat, MatrixCoefficients, PixelRange, PixelType, Size,
                     Ssimulacra2Config, Ssimulacra2Pipeline, TransferCharacteristics)

pytestmark = pytest.mark.gpu

FORMAT = ImageFormat(type=PixelType.Float, family=ColorFamily.Rgb, range=PixelRange.Full, matrix=MatrixCoefficients.Rgb,
                     transfer=TransferCharacteristics.St2084, primaries=ColorPrimaries.Bt2020, depth=32)


@pytest.mark.parametrize("w,h", [(8, 8), (67, 21)])
def test_samples_past_the_curve(w, h):
    rng = np.random.default_rng(w)
    base = (0.2 + 0.5 * rng.random((3, h, w))).astype(np.float32)

    def norms(sample):
        other = base.copy()
        other[:, h // 2, ::3] = sample
        a, b = (Image(Size(w, h), FORMAT, np.ascontiguousarray(x).view(np.uint8).ravel()) for x in (base, other))
        with Ssimulacra2Pipeline(Ssimulacra2Config(size=Size(w, h))) as p:
            return np.asarray(p.Compute(a, b).norms())

    past = norms(3.0)
    assert np.array_equal(norms(5.0), past, equal_nan=True)
    low, high = norms(0.5), norms(0.9)
    assert np.isfinite(low).all() and np.isfinite(high).all()
    assert not np.array_equal(low, past, equal_nan=True) and not np.array_equal(low, high)
