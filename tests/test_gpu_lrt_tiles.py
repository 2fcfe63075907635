"""Local Radon transform at the edges of its tiles (64 columns x 32 rows, 64-cell
blocks of the window sums): sides around 32 and 64, images with and without
empty regions, against the one-thread oracle.  Noise images have no ties of
the peak rule, so every cell agrees to the float32 sum over the sectors; next
to an empty region a window may hold a single pixel row, whose ties the last
bit decides in a few cells."""
import numpy as np
import pytest

import oracle
import skewengine_amd as ske
from skewengine_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2, 3, 31, 32, 33, 63, 64, 65, 97])
@pytest.mark.parametrize("empty", [False, True])
def test_tile_edges_match_oracle(n, empty):
    img = np.random.default_rng(n).uniform(0.1, 1.0, (n, n)).astype(np.float32)
    if empty:
        img[: n // 3] = 0.0
    with ske.SkewEngine(img) as e:
        e.set_option(_lib.OPT_RADON_LOCAL, 1)
        out = e.run(ske.KERNEL_RADON)
    ref, _ = oracle.execute(oracle.RADON_LOCAL, img, nthreads=1)
    # 180 float32 additions of non-negative values: 180 half ulps
    bad = ~np.isclose(out, ref, rtol=180 * 2.0 ** -24, atol=1e-9 * np.abs(ref).max())
    assert bad.mean() <= (5e-3 if empty else 0.0)
