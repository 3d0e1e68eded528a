"""GPU parity: the softmax of a Network layer at the lengths where its sum changes form (a chain
of adds up to 512 active neurons, the windowed exact sum to 8192, passes beyond), vs the
oracle's sequential sum.  Bar: bit-exact."""
import numpy as np
import pytest

from test_gpu_slide_train import build, spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 31, 32, 33, 511, 512, 513, 1025, 8192, 8193, 9000])
def test_softmax_lengths(kh, orc, n):
    rng = np.random.default_rng(n)
    # one table of two buckets that hold every neuron: all n are active
    net, layers, onet = build(orc, [spec(rng, 12, n, "Softmax", sampling="Vanilla", k=1, L=1, cap=1, seed=2)])
    X = np.zeros((2, 12), np.float32)
    X[0] = rng.standard_normal(12)
    for l, ol in zip(layers, onet.layers):     # an empty index: the all-neurons fallback, in id order
        l.index.clear()
        ol["index"].len[:] = 0
    got = net.predict_batch(X).cpu().numpy()
    for i in range(2):
        np.testing.assert_array_equal(got[i], onet.predict(X[i]))
