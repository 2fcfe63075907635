"""Viewshed rows past 4096 cells: blocks of visibility bits whose closed runs
are added one by one, with the early exit, against the kernel that steps every
scan (OPT_SDEM_VARIANT = 2).  The sums pass 2^24, so any other order of the
additions shows.  Terrains with long visible runs (a bowl), none (a cone) and
many (noise, fBm); sides just past 4096 and sectors of every orientation."""
import numpy as np
import pytest

import skewengine_amd as ske
from skewengine_amd import _lib, synth

pytestmark = pytest.mark.gpu


def _terrain(name, n):
    y, x = np.mgrid[0:n, 0:n].astype(np.float32)
    r = np.hypot(x - n / 2, y - n / 3)
    if name == "bowl":
        g = 300.0 * (r / n) ** 2
    elif name == "cone":
        g = 900.0 - 0.2 * r
    elif name == "noise":
        g = np.random.default_rng(n).uniform(0, 30, (n, n))
    else:
        g = synth.dem(n, 0.75, n, 3000.0)
    return np.ascontiguousarray(g, np.float32)


@pytest.mark.parametrize("name,n,povh", [("bowl", 4097, 0.15), ("cone", 4100, 0.15), ("noise", 4159, 3.0),
                                         ("fbm", 4128, 0.15), ("fbm", 5000, 1.2)])
def test_long_rows_match_per_step_kernel(name, n, povh):
    g = _terrain(name, n)
    print("terrain", name, n, flush=True)
    with ske.SkewEngine(g) as e:
        for s0, s1 in [(0, 1), (30, 31), (44, 46), (90, 91), (135, 136), (179, 180)]:
            e.set_option(_lib.OPT_SDEM_VARIANT, 0)
            out = e.run(ske.KERNEL_SDEM, s0, s1, povh=povh)
            e.set_option(_lib.OPT_SDEM_VARIANT, 2)
            assert np.array_equal(out, e.run(ske.KERNEL_SDEM, s0, s1, povh=povh)), (name, n, s0)


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, -3.4028235e38])
def test_long_rows_with_special_heights(value):
    n = 4097
    g = _terrain("fbm", n)
    at = np.random.default_rng(1).integers(0, n, (n * 40, 2))
    g[at[:, 0], at[:, 1]] = value
    with ske.SkewEngine(g) as e:
        for s0 in (0, 61):
            e.set_option(_lib.OPT_SDEM_VARIANT, 0)
            out = e.run(ske.KERNEL_SDEM, s0, s0 + 1)
            e.set_option(_lib.OPT_SDEM_VARIANT, 2)
            assert np.array_equal(out, e.run(ske.KERNEL_SDEM, s0, s0 + 1), equal_nan=True), (value, s0)


@pytest.mark.parametrize("n,s0,s1", [(1100, 0, 180), (2100, 40, 60), (3400, 44, 48), (4300, 44, 46)])
def test_runs_by_row_length_match_per_step_kernel(n, s0, s1):
    """Row lists that cross 1024, 2048, 3328 and 4096 cells, one launch each."""
    g = _terrain("fbm", n)
    with ske.SkewEngine(g) as e:
        out = e.run(ske.KERNEL_SDEM, s0, s1)
        e.set_option(_lib.OPT_SDEM_VARIANT, 2)
        assert np.array_equal(out, e.run(ske.KERNEL_SDEM, s0, s1))


def test_runs_of_an_uneven_batch():
    gs = [_terrain("fbm", n) for n in (150, 1100, 2500, 90)]
    with ske.SkewBatch(gs) as b:
        b.run(ske.KERNEL_SDEM, 30, 60)
        outs = b.outputs()
    for g, out in zip(gs, outs):
        with ske.SkewEngine(g) as e:
            e.set_option(_lib.OPT_SDEM_VARIANT, 2)
            assert np.array_equal(out, e.run(ske.KERNEL_SDEM, 30, 60)), g.shape


@pytest.mark.parametrize("value", [np.nan, np.inf, -np.inf, -3.4028235e38])
def test_rows_with_special_heights_take_the_per_step_scans(value):
    g = synth.dem(128, 0.8, 3, 1500.0)[:100, :100].copy()
    at = np.random.default_rng(1).integers(0, 100, (40, 2))
    g[at[:, 0], at[:, 1]] = value
    with ske.SkewEngine(g) as e:
        out = e.run(ske.KERNEL_SDEM)
        e.set_option(_lib.OPT_SDEM_VARIANT, 2)
        assert np.array_equal(out, e.run(ske.KERNEL_SDEM), equal_nan=True)
