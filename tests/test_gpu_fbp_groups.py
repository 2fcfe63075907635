"""Standard-geometry projector, filter and back-projection over the forms their
dispatch takes: batches of one to nine slices (groups of four, empty slices,
single remainders), sides at the edges of the 67- and 129-pixel projector
tiles and of the 16- and 32-pixel back-projection tiles, detectors at the
edges of the filter's 192 columns and 384-wide chunks.  Every slice must equal
the one-slice result of the same kernels' other form to rounding (a few ulp
of the largest value; the bar of the FP64 tests, 1e-4, is checked on the
first slice)."""
import numpy as np
import pytest

from oracle import std_fbp
from skewengine_amd import synth
from skewengine_amd.fbp import FBP

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nang,ndet,batch", [(16, 3, 25, 2), (66, 5, 95, 3), (67, 4, 192, 4), (128, 7, 193, 5),
                                               (129, 13, 185, 6), (33, 17, 384, 7), (134, 6, 385, 9),
                                               (260, 130, 371, 8)])
def test_batches_equal_single_slices(n, nang, ndet, batch):
    imgs = np.stack([synth.ellipse_phantom(n, seed=b) for b in range(batch)])
    with FBP(n, nang, ndet, max_batch=batch) as f:
        sino = f.radon(imgs)
        rec = f.fbp(sino)
        ref_sino = std_fbp.project(imgs[0], nang, ndet)
        assert np.max(np.abs(sino[0] - ref_sino)) <= 1e-4 * np.max(np.abs(ref_sino))
        ref_rec = std_fbp.fbp(sino[0].astype(np.float64), n)
        assert np.max(np.abs(rec[0] - ref_rec)) <= 1e-4 * np.max(np.abs(ref_rec))
        for b in range(batch):
            # a ray sums at most sqrt(2) n samples of |f| <= 10: float32 sums in another order
            one = f.radon(imgs[b])
            assert np.max(np.abs(sino[b] - one)) <= 64 * 2.0 ** -24 * max(np.max(np.abs(one)), 1.0)
            # the same sinogram row by row: the filter does not depend on the batch, and the
            # back-projection adds the same values in the same order
            assert np.array_equal(rec[b], f.fbp(sino[b]))


@pytest.mark.parametrize("n,batch", [(512, 4), (384, 6)])
def test_four_slice_backprojection_equals_single(n, batch):
    """Sizes whose groups of four take four pixels a thread and one."""
    rng = np.random.default_rng(n)
    nang, ndet = 37, int(1.42 * n)
    sino = rng.standard_normal((batch, nang, ndet)).astype(np.float32)
    with FBP(n, nang, ndet, max_batch=3 * batch) as f:
        wide = f.fbp(np.concatenate([sino] * 3))
        for b in range(batch):
            one = f.fbp(sino[b])
            for k in range(3):
                assert np.array_equal(wide[k * batch + b], one)
