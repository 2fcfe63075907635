"""Radon row sums: how the sectors of a launch are dealt to the eight XCDs (runs
of up to 23, one round of runs for every 184 sectors).  Sector counts at the
edges of the rule, as shares of one grid and as batches of two and three,
against the one-thread oracle bit for bit."""
import numpy as np
import pytest

import oracle
import skewengine_amd as ske

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sides,s0,s1", [((40,), 11, 18), ((40,), 86, 95), ((40,), 40, 56), ((70, 40), 0, 92),
                                         ((70, 40), 3, 96), ((33, 64, 50), 60, 121), ((33, 64, 50), 60, 122),
                                         ((33, 64, 50), 0, 180)])
def test_sector_counts_match_oracle(sides, s0, s1):
    imgs = [np.random.default_rng(n).uniform(0.1, 1.0, (n, n)).astype(np.float32) for n in sides]
    with ske.SkewBatch(imgs) as b:
        b.run(ske.KERNEL_RADON, s0, s1)
        outs = b.outputs()
    for img, out in zip(imgs, outs):
        assert np.array_equal(out, oracle.execute(oracle.RADON, img, nthreads=1, s0=s0, s1=s1)[0])
