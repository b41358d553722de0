"""The prepare kernel's general decode above the split form's 1,024 tiles, over
the input formats: a pair of 1,122 tiles (1041x1043, 1042x1046 and 1044x1048 by
subsampling: the last lane's four columns, the last tile's rows and the last
wave's half are partial) takes the four-row form; scored again with its
original's planes kept, the distorted image's 561 tiles take the split form,
which the format tests hold to FP64 decodes. The samples, and so the norms, are
the same bit for bit, in both places of the pair.
"""
from __future__ import annotations

import numpy as np
import pytest

from vqm_amd import (AlphaType as AT, ChromaFilter, ChromaLocation, ColorFamily as CF, ColorPrimaries as CP, Image,
                     ImageFormat, MatrixCoefficients as MC, PixelRange as PR, PixelType as PT, Size, Ssimulacra2Config,
                     Ssimulacra2Pipeline, TransferCharacteristics as TC, required_bytes)

pytestmark = pytest.mark.gpu


def yuv(type=PT.Byte, sub=(1, 1), matrix=MC.Bt709, transfer=TC.Bt709, primaries=CP.Bt709, depth=8,
        location=ChromaLocation.Left):
    return ImageFormat(type=type, family=CF.Yuv, range=PR.Limited if depth else PR.Full, matrix=matrix,
                       transfer=transfer, primaries=primaries, subsample_w=sub[0], subsample_h=sub[1], depth=depth,
                       chroma_location=location)


HDR = dict(type=PT.Word, depth=10, matrix=MC.Bt2020Ncl, primaries=CP.Bt2020)
FORMATS = {
    "rgb16": ImageFormat(type=PT.Word, depth=16),
    "rgbf32": ImageFormat(),
    "rgbf32 linear": ImageFormat(transfer=TC.Linear),
    "rgbf16": ImageFormat(type=PT.Half),
    "rgba8 straight": ImageFormat(type=PT.Byte, alpha=AT.Straight),
    "rgbaf32 premultiplied": ImageFormat(alpha=AT.Premultiplied),
    "grey8": ImageFormat(type=PT.Byte, family=CF.Grey, matrix=MC.Unspecified, transfer=TC.Bt709),
    "grey12 alpha": ImageFormat(type=PT.Word, depth=12, family=CF.Grey, alpha=AT.Straight, matrix=MC.Unspecified,
                                transfer=TC.Bt709),
    "yuv444p8": yuv(sub=(0, 0)),
    "yuv444f32": yuv(type=PT.Float, depth=0, sub=(0, 0)),
    "yuv422p10": yuv(type=PT.Word, depth=10, sub=(1, 0)),
    "yuv440p8": yuv(sub=(0, 1)),
    "yuv420f16": yuv(type=PT.Half, depth=0),
    "yuv411p8": yuv(sub=(2, 0)),
    "yuv410p8 centre": yuv(sub=(2, 2), location=ChromaLocation.Center),
    "pq420p10": yuv(**HDR, transfer=TC.St2084, location=ChromaLocation.TopLeft),
    "hlg420p10": yuv(**HDR, transfer=TC.AribB67),
    "cl420p10": yuv(**(HDR | dict(matrix=MC.Bt2020Cl))),
    "ictcp420p10": yuv(**(HDR | dict(matrix=MC.Bt2100ICtCp)), transfer=TC.St2084),
    "ycgco444p8": yuv(sub=(0, 0), matrix=MC.YCgCo),
    "log100": ImageFormat(type=PT.Byte, transfer=TC.Log100),
    "log316": ImageFormat(type=PT.Byte, transfer=TC.Log316),
    "xvycc": ImageFormat(type=PT.Byte, transfer=TC.Iec61966_2_4),
    "bt1361": ImageFormat(type=PT.Byte, transfer=TC.Bt1361),
    "st428": ImageFormat(type=PT.Byte, transfer=TC.St428),
    "bt470m": ImageFormat(type=PT.Byte, transfer=TC.Bt470M, primaries=CP.Bt470M),
    "bt470bg": ImageFormat(type=PT.Byte, transfer=TC.Bt470Bg, primaries=CP.Bt470Bg),
}


def image(fmt: ImageFormat, size: Size, seed: int) -> Image:
    n, rng = required_bytes(fmt, size), np.random.default_rng(seed)
    if fmt.type == PT.Byte:
        data = rng.integers(30, 220, n).astype(np.uint8)
    elif fmt.type == PT.Word:
        data = rng.integers(int(0.1 * 2 ** fmt.depth), int(0.85 * 2 ** fmt.depth), n // 2).astype(np.uint16)
    else:
        data = rng.uniform(0.02, 0.6, n // (2 if fmt.type == PT.Half else 4))
        data = data.astype(np.float16 if fmt.type == PT.Half else np.float32)
    return Image(size, fmt, data.view(np.uint8))


def check(fmt: ImageFormat, other: ImageFormat, **cfg):
    """Both forms agree on `fmt` as the distorted and as the original image."""
    side = 1 << max(fmt.subsample_w, fmt.subsample_h)
    size = Size(*{1: (1041, 1043), 2: (1042, 1046), 4: (1044, 1048)}[side])
    with Ssimulacra2Pipeline(Ssimulacra2Config(size=size, gpu_resident_images=2, **cfg)) as p:
        a, b = p.Upload(image(other, size, 1)), p.Upload(image(fmt, size, 2))
        for first, second in ((a, b), (b, a)):
            both = np.asarray(p.Compute(first, second).norms())
            assert p.PreparedImages() == 2
            again = np.asarray(p.Compute(first, second).norms())
            assert p.PreparedImages() == 1
            assert np.isfinite(both).all() and both.any()
            np.testing.assert_array_equal(again, both)


@pytest.mark.parametrize("name", list(FORMATS))
def test_formats(name):
    print(name, flush=True)
    fmt = FORMATS[name]
    subsampled = fmt.subsample_w or fmt.subsample_h
    for flt in ChromaFilter if subsampled else [ChromaFilter.Bilinear]:
        check(fmt, fmt, chroma_filter=int(flt))


@pytest.mark.parametrize("planes", [1, 2, 3])
@pytest.mark.parametrize("name", ["yuv420f16", "pq420p10", "rgba8 straight"])
def test_plane_formats(name, planes):
    check(FORMATS[name], FORMATS[name], plane_format=planes)
    check(FORMATS[name], FORMATS[name], plane_format=planes, map_form=2)


@pytest.mark.parametrize("name", ["rgbf32", "yuv411p8", "hlg420p10"])
def test_beside_a_table_image(name):
    check(FORMATS[name], ImageFormat.srgb8(), chroma_filter=int(ChromaFilter.Lanczos))
