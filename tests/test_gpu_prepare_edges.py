"""The prepare kernel's tiles where their edges fall: a wave takes 64 x 16
base pixels, a lane 4 x 4, rows are loaded four bytes at a time at any
alignment, and levels 3 and 4 share a pass.

Table decode: bit-level with the oracle (1e-10, the order of the FP64 sums;
see test_gpu_scale_parts.py). General decode: the same samples as bytes,
as 16-bit words of the same depth and as the floats they decode to take
different loads (four samples at once, one at a time) and the same arithmetic
from there, so their norms are equal bit for bit.
"""
from __future__ import annotations

import numpy as np
import pytest

import format_ref as fr
import vqm_amd
from conftest import random_pair
from vqm_amd import (AlphaType, ColorFamily, ColorPrimaries, Image, ImageFormat, MapForm, MatrixCoefficients,
                     PixelRange, PixelType, Size, Ssimulacra2Config, Ssimulacra2Pipeline, TransferCharacteristics)

pytestmark = pytest.mark.gpu

SIZES = [(61, 15), (64, 16), (65, 17), (67, 31), (130, 33), (253, 250), (257, 261), (66, 129)]


@pytest.mark.parametrize("planes,map_form", [(vqm_amd.PLANES_F32, MapForm.Reference),
                                             (vqm_amd.PLANES_F16, MapForm.Reference),
                                             (vqm_amd.PLANES_U16, MapForm.Difference)])
def test_table_tiles_at_their_edges(oracle_lib, planes, map_form):
    for i, (w, h) in enumerate(SIZES):
        print(f"prepare {w}x{h} planes {planes}", flush=True)
        a, b = random_pair(w, h, seed=500 + i)
        with Ssimulacra2Pipeline(Ssimulacra2Config(size=Size(w, h), plane_format=planes, map_form=map_form)) as p:
            got = p.Compute(Image(Size(w, h), ImageFormat.srgb8(), a), Image(Size(w, h), ImageFormat.srgb8(), b)).norms()
        _, want, _ = oracle_lib.compute(oracle_lib.form_for(planes, int(map_form)), w, h, a, b)
        np.testing.assert_allclose(got, want, rtol=1e-10, atol=0)


def general(pixel, family, alpha=AlphaType.NoAlpha):
    yuv = family == ColorFamily.Yuv
    return ImageFormat(type=pixel, family=family, alpha=alpha, range=PixelRange.Limited if yuv else PixelRange.Full,
                       matrix=MatrixCoefficients.Bt709 if yuv else
                       MatrixCoefficients.Unspecified if family == ColorFamily.Grey else MatrixCoefficients.Rgb,
                       transfer=TransferCharacteristics.Bt709, primaries=ColorPrimaries.Bt709,
                       depth=0 if pixel == PixelType.Float else 8)


@pytest.mark.parametrize("family,alpha", [(ColorFamily.Yuv, AlphaType.NoAlpha), (ColorFamily.Rgb, AlphaType.Straight),
                                          (ColorFamily.Grey, AlphaType.NoAlpha)])
def test_general_loads_at_any_alignment(family, alpha):
    for i, (w, h) in enumerate(SIZES):
        print(f"general {w}x{h} family {int(family)}", flush=True)
        rng = np.random.default_rng(600 + i)
        size = Size(w, h)
        codes = [{p: rng.integers(16, 236, (h, w)) for p, _, _ in fr.plane_shapes(general(PixelType.Byte, family, alpha), size)}
                 for _ in range(2)]
        norms = []
        for pixel in (PixelType.Byte, PixelType.Word, PixelType.Float):
            fmt = general(pixel, family, alpha)
            byte = general(PixelType.Byte, family, alpha)
            images = []
            for planes in codes:
                parts = []
                for p, _, _ in fr.plane_shapes(fmt, size):
                    if pixel == PixelType.Float:
                        # The decode's own FP32 multiplication and addition.
                        scale, offset = vqm_amd.plane_scale_offset(byte, chroma=p in (1, 2) and family == ColorFamily.Yuv,
                                                                   alpha=p == 3)
                        raw = planes[p].astype(np.float32) * np.float32(scale) + np.float32(offset)
                    else:
                        raw = planes[p].astype(np.uint8 if pixel == PixelType.Byte else np.uint16)
                    data = raw.tobytes()
                    parts.append(data + b"\0" * (-len(data) % 4))
                images.append(Image(size, fmt, np.frombuffer(b"".join(parts), np.uint8)))
            with Ssimulacra2Pipeline(Ssimulacra2Config(size=size)) as p:
                norms.append(p.Compute(*images).norms())
        assert norms[0].any()
        np.testing.assert_array_equal(norms[1], norms[0])
        np.testing.assert_array_equal(norms[2], norms[0])
