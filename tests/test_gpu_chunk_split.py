"""Where the sectors of a grid are cut into chunks must not show.  The maximum
of the cepstrum's deskew reads, for the 90 degree sector, the row that the
sector before it left behind, so these two stay in one chunk: whole runs
against runs with a small arena and against the run in the static scratch
array, for ranges that begin at every sector shortly before 90."""
import numpy as np
import pytest

import skewengine_amd as ske
from skewengine_amd import _lib, synth

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def _whole(img, s0, s1, arena=None):
    with ske.SkewEngine(img) as e:
        if arena:
            e.set_option(_lib.OPT_ARENA_BYTES, arena)
        return e.run(ske.KERNEL_CEPSTRUM, s0, s1)


def test_small_arena():
    img = synth.blurred_texture(200, 0.6, seed=1)[0]
    for s0 in range(76, 91):
        assert np.array_equal(_whole(img, s0, 94), _whole(img, s0, 94, arena=1 << 20)), s0


def test_small_arena_of_a_batch():
    imgs = [synth.blurred_texture(n, 0.6, seed=n)[0] for n in (150, 200, 120)]
    for s0 in range(76, 91):
        with ske.SkewBatch(imgs) as b:
            b.run(ske.KERNEL_CEPSTRUM, s0, 94)
            ref = b.outputs()
        with ske.SkewBatch(imgs) as b:
            b.set_option(_lib.OPT_ARENA_BYTES, 1 << 20)
            b.run(ske.KERNEL_CEPSTRUM, s0, 94)
            for x, y in zip(ref, b.outputs()):
                assert np.array_equal(x, y), s0


def test_scratch_array():
    n = 1000
    img = synth.blurred_texture(n, 0.6, seed=2)[0]
    d_in = torch.from_numpy(img).cuda()
    d_out = torch.zeros(n, n, device="cuda")
    torch.cuda.synchronize()
    for s0 in range(60, 90):
        _lib.check(_lib.lib().ske_execute_noalloc(ske.KERNEL_CEPSTRUM, n, d_in.data_ptr(), d_out.data_ptr(), 0.15, s0,
                                                  92, 0, None))
        assert np.array_equal(d_out.cpu().numpy(), _whole(img, s0, 92)), s0
