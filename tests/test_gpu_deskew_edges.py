"""Deskew and reduce at the edges of their blocks (16 or 4 output rows a
thread, 256 columns a workgroup, 32 x 32 reduce tiles), in one chunk and with
an orientation's sectors spread over several: against the one-thread oracle
where the operator is bit-exact, and against the per-sector calls otherwise."""
import numpy as np
import pytest

import oracle
import skewengine_amd as ske
from skewengine_amd import _lib, synth

pytestmark = pytest.mark.gpu

SIDES = [2, 3, 4, 5, 15, 16, 17, 31, 33, 48, 255, 256, 257, 275]


@pytest.mark.parametrize("n", SIDES)
@pytest.mark.parametrize("arena", [0, 1 << 20])
def test_viewshed_edges_match_oracle(n, arena):
    g = synth.dem(64 * -(-n // 64), 0.8, n, 1500.0)[:n, :n].copy()
    ref, _ = oracle.execute(oracle.SDEM, g, nthreads=1)
    with ske.SkewEngine(g) as e:
        if arena:
            e.set_option(_lib.OPT_ARENA_BYTES, arena)
        for _ in range(2):  # the second run must not see the first's sums
            assert np.array_equal(e.run(ske.KERNEL_SDEM), ref)


@pytest.mark.parametrize("s0,s1", [(0, 1), (45, 46), (90, 91), (135, 136), (40, 50), (89, 137)])
def test_few_sectors_match_oracle(s0, s1):
    g = synth.dem(64, 0.8, 7, 1500.0)[:50, :50].copy()
    with ske.SkewEngine(g) as e:
        e.run(ske.KERNEL_SDEM)  # leaves every orientation's sums behind
        out = e.run(ske.KERNEL_SDEM, s0, s1)
    assert np.array_equal(out, oracle.execute(oracle.SDEM, g, nthreads=1, s0=s0, s1=s1)[0])


@pytest.mark.parametrize("n", [2, 7, 50, 62, 63, 64, 131, 190])
@pytest.mark.parametrize("s0,s1", [(0, 180), (0, 1), (45, 46), (3, 25), (3, 26), (80, 104), (1, 180), (0, 8)])
def test_radon_sector_ranges_match_oracle(n, s0, s1):
    """Row sums around 63 rows a wave, sector counts around the runs of 23 that share an XCD; filters of 2 to 512
    points."""
    img = np.random.default_rng(n).uniform(0.1, 1.0, (n, n)).astype(np.float32)
    with ske.SkewEngine(img) as e:
        out = e.run(ske.KERNEL_RADON, s0, s1)
    assert np.array_equal(out, oracle.execute(oracle.RADON, img, nthreads=1, s0=s0, s1=s1)[0])


def _per_sector(e, kernel, is_max, n):
    e.set_kernel(kernel, 0.15)
    for a in range(180):
        e.skew(a)
        e.kernel()
        e.deskew(is_max)
    return e.reduce(np.zeros((n, n), np.float32), is_max)


@pytest.mark.parametrize("n", SIDES)
@pytest.mark.parametrize("kernel,is_max", [(ske.KERNEL_CEPSTRUM, 1), (ske.KERNEL_RADON, 0)])
def test_run_equals_per_sector_calls(n, kernel, is_max):
    img = np.random.default_rng(n).uniform(0.1, 1.0, (n, n)).astype(np.float32)
    with ske.SkewEngine(img) as e, ske.SkewEngine(img) as f:
        out = e.run(kernel)
        if is_max:  # in one chunk: a chunk's first sector has no predecessor whose row the maximum could see
            assert np.array_equal(out, _per_sector(f, kernel, is_max, n))
        else:  # the row sums are added in another order there
            ref = _per_sector(f, kernel, is_max, n)
            assert np.max(np.abs(out - ref)) <= 1e-6 * np.max(np.abs(ref))


def test_staged_radon_of_a_batch_equals_single_images():
    """More than 1024 workgroups: the staged kernel; alone, each image takes the other one."""
    sides = SIDES + [64] * 80 + [300, 257, 511, 300]
    rng = np.random.default_rng(3)
    imgs = [rng.uniform(0.0, 1.0, (n, n)).astype(np.float32) for n in sides]
    with ske.SkewBatch(imgs) as b:
        b.run(ske.KERNEL_RADON)
        outs = b.outputs()
    for n, img, out in list(zip(sides, imgs, outs))[:len(SIDES) + 1] + list(zip(sides, imgs, outs))[-4:]:
        with ske.SkewEngine(img) as e:
            assert np.array_equal(out, e.run(ske.KERNEL_RADON)), n
