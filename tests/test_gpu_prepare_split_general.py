"""The prepare kernel's two forms in the general decode (split up to 1,024
tiles): a pair of 1,080 tiles takes the other form, and scored again with its
original's planes kept, 540 tiles, the split form for the distorted image. The
samples, and so the norms, are the same bit for bit.
"""
from __future__ import annotations

import numpy as np
import pytest

from vqm_amd import (ColorFamily, ColorPrimaries, Image, ImageFormat, MatrixCoefficients, PixelRange, PixelType, Size,
                     Ssimulacra2Config, Ssimulacra2Pipeline, TransferCharacteristics)

pytestmark = pytest.mark.gpu

FORMATS = {
    "yuv420p8": ImageFormat(type=PixelType.Byte, family=ColorFamily.Yuv, range=PixelRange.Limited,
                            matrix=MatrixCoefficients.Bt709, transfer=TransferCharacteristics.Bt709,
                            primaries=ColorPrimaries.Bt709, subsample_w=1, subsample_h=1),
    "pq420p10": ImageFormat(type=PixelType.Word, family=ColorFamily.Yuv, range=PixelRange.Limited,
                            matrix=MatrixCoefficients.Bt2020Ncl, transfer=TransferCharacteristics.St2084,
                            primaries=ColorPrimaries.Bt2020, subsample_w=1, subsample_h=1, depth=10),
}


@pytest.mark.parametrize("name", list(FORMATS))
@pytest.mark.parametrize("chroma_filter", [0, 1])
@pytest.mark.parametrize("planes", [0, 3])
def test_forms_agree(name, chroma_filter, planes):
    w, h, f = 1276, 862, FORMATS[name]
    rng = np.random.default_rng(7)
    # Planes start on 4-byte boundaries.
    scale = 1 if f.type == PixelType.Byte else 2
    sizes = [-(-n * scale // 4) * 4 for n in (w * h, w * h // 4, w * h // 4)]

    def image():
        low, high = (60, 180) if scale == 1 else (300, 700)
        kind = np.uint8 if scale == 1 else np.uint16
        return Image(Size(w, h), f, rng.integers(low, high, sum(sizes) // scale).astype(kind).view(np.uint8))

    cfg = Ssimulacra2Config(size=Size(w, h), gpu_resident_images=2, chroma_filter=chroma_filter, plane_format=planes)
    with Ssimulacra2Pipeline(cfg) as p:
        a, b = p.Upload(image()), p.Upload(image())
        both = np.asarray(p.Compute(a, b).norms())
        again = np.asarray(p.Compute(a, b).norms())
    assert both.any()
    np.testing.assert_array_equal(again, both)
