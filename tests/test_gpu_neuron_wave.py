"""Training steps through a wave per neuron, bit for bit against the oracle: rows with 1,
63..65, 255..257 and all nonzeros, layers of 130 to 2000 inputs (row-major, not the
32-neuron tiles), one to seventy neurons."""
import numpy as np
import pytest

from test_gpu_slide_train import build, run_steps, spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,hidden", [(130, 1), (300, 5), (2000, 70), (257, 131)])
def test_train_over_entry_counts(kh, orc, dim, hidden):
    rng = np.random.default_rng(dim)
    counts = sorted({min(c, dim) for c in (1, 15, 16, 17, 63, 64, 65, 255, 256, 257, dim)})
    X = np.zeros((len(counts), dim), np.float32)
    for x, c in zip(X, counts):
        x[rng.choice(dim, c, replace=False)] = rng.normal(0, 1, c)
    labels = [sorted(rng.choice(6, 1 + i % 2, replace=False).tolist()) for i in range(len(X))]
    net, layers, onet = build(orc, [spec(rng, dim, hidden, "Relu", top_k=hidden), spec(rng, hidden, 6, "Softmax", top_k=6)])
    run_steps(net, layers, onet, X, labels, 0.01, 2, len(X))
