"""The CPU check of the projector's tile bounds (test_projector_tiles.py) at the
tile side that batches take: four slices a workgroup, tiles of up to 67 base
pixels (kPtMax4 in skewengine_amd/csrc/fbp.h) instead of 129 (kPtMax1)."""
import math
import os
import re

import numpy as np
import pytest

import test_projector_tiles as tiles

HEADER = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "skewengine_amd", "csrc", "fbp.h")


def _sides():
    with open(HEADER) as f:
        m = re.search(r"kPtMax1 = (\d+), kPtMax4 = (\d+);", f.read())
    return int(m.group(1)), int(m.group(2))


@pytest.fixture
def four_slices(monkeypatch):
    one, four = _sides()
    assert one == tiles.KPT_MAX
    monkeypatch.setattr(tiles, "KPT_MAX", four)
    return four


@pytest.mark.parametrize("n", [2, 31, 65, 66, 67, 68, 100, 133, 134, 200])
def test_tile_bounds(four_slices, n):
    rng = np.random.default_rng(n)
    angles = [a * math.pi / 4 for a in range(8)] + [math.pi * a / 24 for a in range(24)] + list(rng.uniform(-10, 10, 4))
    for ndet in sorted({2, n, int(1.4143 * n) + 1, 2 * n + 3}):
        for th in angles:
            tiles._check_angle(n, ndet, th)


def test_tiling_covers_the_base_pixels(four_slices):
    for n in list(range(1, 600)) + [1023, 1024, 2048, 8192]:
        ntx, ts, _ = tiles.proj_tiling(n)
        assert 1 <= ts <= four_slices and ntx * ts >= n + 1 and (ntx - 1) * ts < n + 1
