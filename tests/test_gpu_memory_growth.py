"""Host memory does not grow with the pairs scored: the runtime must release
each submission's commands and events.

Bound: 2,000 submissions that kept their commands would hold 4.9 KB each, 9.8
MB; half of that is allowed, which the allocator's own growth (below 0.5 MB
measured) stays far from.
"""
from __future__ import annotations

import pytest

from conftest import random_pair
from vqm_amd import (DeviceBuffer, DeviceImage, Image, ImageFormat, Size, Ssimulacra2Batch, Ssimulacra2Config,
                     Ssimulacra2Pipeline)

pytestmark = pytest.mark.gpu

W, H, RUNS, BOUND = 96, 64, 2000, 4 << 20


def resident_bytes() -> int:
    with open("/proc/self/statm") as f:
        return int(f.read().split()[1]) * 4096


def growth(step) -> int:
    for _ in range(200):
        step()
    before = resident_bytes()
    for _ in range(RUNS):
        step()
    return resident_bytes() - before


@pytest.fixture(scope="module")
def pair():
    a, b = random_pair(W, H, seed=5)
    da, db = DeviceBuffer(a.nbytes), DeviceBuffer(b.nbytes)
    da.upload(a)
    db.upload(b)
    return a, b, da, db


@pytest.mark.parametrize("source", ["device", "host", "graph"])
def test_pipeline(pair, source):
    a, b, da, db = pair
    f, size = ImageFormat.srgb8(), Size(W, H)
    x = Image(size, f, a) if source == "host" else DeviceImage(da.ptr, size, f)
    y = Image(size, f, b) if source == "host" else DeviceImage(db.ptr, size, f)
    with Ssimulacra2Pipeline(Ssimulacra2Config(size=size, graph=source == "graph")) as p:
        assert growth(lambda: p.Compute(x, y)) < BOUND


@pytest.mark.parametrize("graph", [False, True])
def test_batch(pair, graph):
    _, _, da, db = pair
    items = [(da.ptr, db.ptr, W, H)] * 2
    batch = Ssimulacra2Batch(2, graph=graph)
    grown = growth(lambda: batch.Finish(batch.Submit(items), raw=True))
    batch.close()
    assert grown < BOUND
