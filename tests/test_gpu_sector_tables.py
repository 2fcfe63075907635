"""The per-sector calls' table ring: more sectors than slots without a wait
between them, sides whose ring has 16 and 2 slots, and several engines in turn;
each sector's result against the all-sector run of that sector alone."""
import ctypes

import numpy as np
import pytest
import torch

import skewengine_amd as ske
from skewengine_amd import synth
from skewengine_amd._lib import check, lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,angles", [(2, range(180)), (50, range(179, -1, -1)), (301, range(0, 180, 4)),
                                      (2100, (0, 44, 45, 46, 91, 134, 179))])
def test_sectors_without_waits_equal_the_run(n, angles):
    g = synth.dem(64 * -(-n // 64), 0.8, n, 1500.0)[:n, :n].copy()
    with ske.SkewEngine(g) as e, ske.SkewEngine(g) as f, ske.SkewEngine(g) as r:
        e.set_kernel(ske.KERNEL_IDENTITYDEM)
        f.set_kernel(ske.KERNEL_IDENTITYDEM)
        ref = np.zeros((n, n), np.float64)
        for a in angles:
            for x in (e, f):
                x.skew(a)
                x.kernel()
                x.deskew()
            ref += r.run(ske.KERNEL_IDENTITYDEM, a, a + 1)
        out = e.reduce(np.zeros((n, n), np.float32))
        assert np.array_equal(out, f.reduce(np.zeros((n, n), np.float32)))
    # one float32 addition per sector and orientation, of non-negative values
    assert np.allclose(out, ref, rtol=(len(list(angles)) + 4) * 2.0 ** -24, atol=0)


def test_tables_of_the_last_sector():
    g = synth.dem(64, 0.8, 1, 1500.0)
    with ske.SkewEngine(g) as e:
        e.set_kernel(ske.KERNEL_IDENTITYDEM)
        for a in range(40):
            e.skew(a)
        e.kernel()
        S, SO = e.skew_buffers()
        _, t, w, f, l = ske.plan_sector(64, 64, 39)
        for r in range(S.shape[0]):
            j = np.arange(f[r], l[r])
            assert np.array_equal(SO[r, j], S[r, j]) and not SO[r, :f[r]].any() and not SO[r, l[r]:].any()


@pytest.mark.parametrize("before", [True, False])
def test_device_operator_finds_the_sector_ready(before):
    """An operator may read skewInput on a stream of its own: the engine's is
    idle when it is called, whether it was set before or after skew()."""
    form = ctypes.CFUNCTYPE(None, ctypes.c_void_p, ctypes.c_void_p, ctypes.c_int, ctypes.c_int, ctypes.c_void_p,
                            ctypes.c_void_p, ctypes.c_float, ctypes.c_int, ctypes.c_void_p, ctypes.c_void_p)
    idle = []
    op = form(lambda so, s, dim_i, h, last, first, val, angle, stream, user:
              idle.append(torch.cuda.ExternalStream(stream).query()))
    with ske.SkewEngine(synth.dem(1024, 0.8, 3, 1500.0)) as e:
        if before:
            check(lib().ske_set_device_operator(e._h, ctypes.cast(op, ctypes.c_void_p), None))
        for a in range(12):
            e.skew(a)
        if not before:
            check(lib().ske_set_device_operator(e._h, ctypes.cast(op, ctypes.c_void_p), None))
        e.kernel()
    assert idle == [True]
