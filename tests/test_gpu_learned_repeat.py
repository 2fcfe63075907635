"""The CNN's gradients are sums in a fixed order: two passes on the same input
give the same bits (weights and biases of every layer; the filter taps are
added with float atomics and left out)."""
import numpy as np
import pytest

from oracle import learned_ref as L
from skewengine_amd import learned as lm
from skewengine_amd.fbp import FBP
from test_gpu_learned import _random_params

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,batch,channels", [(32, 1, 16), (256, 6, 16), (256, 3, 32), (512, 8, 16)])
def test_two_passes_give_the_same_cnn_gradients(n, batch, channels):
    with FBP(n, 6, n, max_batch=batch) as f, lm.LearnedFBP(f, channels=channels) as m:
        m.set_params(_random_params(m, n, n, seed=3))
        m.make_batch(batch, seed=7, i0=1e4, mu=1.0)
        loss, grad = m.gradient(batch)
        first = np.array(grad)[:L.layout(channels)[1]]
        for _ in range(8):
            again, grad = m.gradient(batch)
            assert again == loss
            assert np.array_equal(np.array(grad)[:L.layout(channels)[1]], first)
