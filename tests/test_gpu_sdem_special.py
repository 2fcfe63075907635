"""Viewshed of grids with heights (or an observer height) that are not finite or
are huge, through every launch shape of the bit-block kernels and call by call:
the sign of a difference is not its comparison there, so such rows take the
per-step scans and equal OPT_SDEM_VARIANT = 2, and with it the one-thread oracle
(quotients of infinite differences, the running maximum with a quotient that is
no number), bit for bit."""
import numpy as np
import pytest

import oracle
import skewengine_amd as ske
from skewengine_amd import _lib, synth

pytestmark = pytest.mark.gpu

SHAPES = {"default": {}, "group 1": {_lib.OPT_SDEM_GROUP: 1},
          "group 1, 2 waves": {_lib.OPT_SDEM_GROUP: 1, _lib.OPT_SDEM_WAVES: 2},
          "group 1, 8 waves": {_lib.OPT_SDEM_GROUP: 1, _lib.OPT_SDEM_WAVES: 8},
          "persistent": {_lib.OPT_SDEM_PERSISTENT: 8},
          "persistent, group 1": {_lib.OPT_SDEM_PERSISTENT: 8, _lib.OPT_SDEM_GROUP: 1}}


def _grid(value=None, n=100):
    g = synth.dem(128, 0.8, 3, 1500.0)[:n, :n].copy()
    if value is not None:
        at = np.random.default_rng(1).integers(0, n, (40, 2))
        g[at[:, 0], at[:, 1]] = value
    return g


def _per_step(g, povh):
    with ske.SkewEngine(g) as e:
        e.set_option(_lib.OPT_SDEM_VARIANT, 2)
        return e.run(ske.KERNEL_SDEM, povh=povh)


def _by_calls(g, povh, variant):
    with ske.SkewEngine(g) as e:
        e.set_option(_lib.OPT_SDEM_VARIANT, variant)
        e.set_kernel(ske.KERNEL_SDEM, povh)
        for a in range(180):
            e.skew(a)
            e.kernel()
            e.deskew()
        return e.reduce(np.zeros_like(g))


CASES = [(v, 0.15) for v in (np.nan, np.inf, -np.inf, -3.4028235e38, 3.4028235e38)]
CASES += [(None, p) for p in (np.nan, np.inf, -np.inf, 3.4028235e38)]


@pytest.mark.parametrize("shape", SHAPES)
@pytest.mark.parametrize("value,povh", CASES)
def test_launch_shapes_equal_the_per_step_scans(value, povh, shape):
    g = _grid(value)
    ref = _per_step(g, povh)
    with ske.SkewEngine(g) as e:
        for option, v in SHAPES[shape].items():
            e.set_option(option, v)
        assert np.array_equal(e.run(ske.KERNEL_SDEM, povh=povh), ref, equal_nan=True)


@pytest.mark.parametrize("value,povh", CASES)
def test_calls_equal_the_per_step_scans(value, povh):
    g = _grid(value, 60)
    assert np.array_equal(_by_calls(g, povh, 0), _by_calls(g, povh, 2), equal_nan=True)


@pytest.mark.parametrize("variant", [0, 1, 2])
@pytest.mark.parametrize("value,povh", CASES)
def test_variants_equal_the_oracle(value, povh, variant):
    g = _grid(value)
    with ske.SkewEngine(g) as e:
        e.set_option(_lib.OPT_SDEM_VARIANT, variant)
        out = e.run(ske.KERNEL_SDEM, povh=povh)
    assert np.array_equal(out, oracle.execute(oracle.SDEM, g, nthreads=1, povh=povh)[0], equal_nan=True)


@pytest.mark.parametrize("value,povh", CASES)
def test_scratch_array_equals_the_oracle(value, povh):
    torch = pytest.importorskip("torch")
    g = _grid(value)
    d_in, d_out = torch.from_numpy(g).cuda(), torch.empty(g.shape, device="cuda")
    torch.cuda.synchronize()
    _lib.check(_lib.lib().ske_execute_noalloc(ske.KERNEL_SDEM, g.shape[0], d_in.data_ptr(), d_out.data_ptr(), povh, 0,
                                              180, 0, None))
    assert np.array_equal(d_out.cpu().numpy(), oracle.execute(oracle.SDEM, g, nthreads=1, povh=povh)[0], equal_nan=True)
