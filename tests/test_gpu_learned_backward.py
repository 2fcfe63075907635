"""Training gradients of the learned FBP at the edges of the backward kernels'
work split, against the FP64 oracle: images of 2 x 2 and 5 x 5 tiles, batches
that leave slices of a group of four empty, sides whose adjoint runs in one
and in two shares of lines, detectors that are no multiple of the filter
gradient's eight lags.  Bars as in test_gpu_learned.py (fp32 sums: 2e-4 of a
layer's largest weight gradient, 1e-4 of the largest adjoint and tap value)."""
import numpy as np
import pytest

from oracle import learned_ref as L
from skewengine_amd import learned as lm
from skewengine_amd.fbp import FBP, IMAGE, RECON, SINO
from test_gpu_learned import _bf, _random_params, _rel

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,nang,ndet,batch,channels", [(32, 7, 46, 1, 16), (32, 5, 48, 5, 32), (96, 9, 131, 4, 16),
                                                        (160, 6, 229, 2, 32), (160, 11, 233, 3, 16)])
def test_gradients_at_split_edges(n, nang, ndet, batch, channels):
    with FBP(n, nang, ndet, max_batch=batch) as f, lm.LearnedFBP(f, channels=channels) as m:
        prm = _random_params(m, ndet, n, seed=5 + n)
        m.set_params(prm)
        m.make_batch(batch, seed=17, i0=1e4, mu=1.0)
        sino, target = f.download(SINO, batch), f.download(IMAGE, batch)
        _, grad = m.gradient(batch)
        out, r0 = f.download(RECON, batch), m.download(lm.R0, batch)
        acts = [_bf(m.download(w, batch)) for w in (lm.A1, lm.A2, lm.A3)]
        dr0, dq = m.download(lm.DR0, batch), m.download(lm.FILTERED_GRAD, batch)
    p64 = prm.astype(np.float64)
    dout = 2.0 * (out.astype(np.float64) - target) / target.size
    cache = {"x0": L.bf16(r0)[..., None], "a1": acts[0], "a2": acts[1], "a3": acts[2]}
    off, taps_off = L.layout(channels)
    ref, ref_dr0 = L.cnn_backward(p64, cache, dout, C=channels)
    for name, (o, s) in off.items():
        assert _rel(grad[o:o + s], np.asarray(ref[name]).reshape(-1)) <= 2e-4, name
    assert _rel(dr0, ref_dr0) <= 1e-4
    ref_dq = np.stack([L.backproject_adjoint(dr0[b], nang, ndet) for b in range(batch)])
    assert _rel(dq, ref_dq) <= 1e-4
    dfull = sum(L.filter_grad(ref_dq[b], sino[b]) for b in range(batch))
    assert _rel(grad[taps_off:], L.fold_taps(dfull)) <= 1e-4


@pytest.mark.parametrize("n,channels", [(544, 16), (384, 32)])
def test_weight_gradients_past_one_tile_a_workgroup(n, channels):
    """34^2 and 24^2 tiles: a few more than the workgroups that go through
    them, so some take a second tile and most none."""
    with FBP(n, 3, n, max_batch=1) as f, lm.LearnedFBP(f, channels=channels) as m:
        prm = _random_params(m, n, n, seed=11)
        m.set_params(prm)
        m.make_batch(1, seed=3, i0=1e4, mu=1.0)
        target = f.download(IMAGE, 1)
        _, grad = m.gradient(1)
        out, r0 = f.download(RECON, 1), m.download(lm.R0, 1)
        acts = [_bf(m.download(w, 1)) for w in (lm.A1, lm.A2, lm.A3)]
    dout = 2.0 * (out.astype(np.float64) - target) / target.size
    cache = {"x0": L.bf16(r0)[..., None], "a1": acts[0], "a2": acts[1], "a3": acts[2]}
    ref, _ = L.cnn_backward(prm.astype(np.float64), cache, dout, C=channels)
    for name, (o, s) in L.layout(channels)[0].items():
        assert _rel(grad[o:o + s], np.asarray(ref[name]).reshape(-1)) <= 2e-4, name
