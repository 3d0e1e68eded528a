"""SLIDE forward, bit for bit against the oracle, at the edges of its entry lists: rows
with 0, 1 and around 16, 32 and all dimensions nonzero; dimensions around a load of a
block (256) and of four (1024), the 32-neuron tiles (dimensions up to 128, a multiple
of 4; fewer than one, of four waves and of eight) and the largest dense input; row-major and transposed weights (act); sparse
inputs longer than the list kept on chip (4096)."""
import numpy as np
import pytest

from test_gpu_lsh_slide import FIFO, check_slide, slide_pair

pytestmark = pytest.mark.gpu


def rows_of(rng, dim):
    counts = sorted({min(c, dim) for c in (0, 1, 15, 16, 17, 31, 32, 33, 64, 65, dim - 1, dim)})
    X = np.zeros((len(counts), dim), np.float32)
    for x, c in zip(X, counts):
        x[rng.choice(dim, c, replace=False)] = rng.normal(0, 1, c)
    return X


@pytest.mark.parametrize("dim,n", [(4, 1), (128, 31), (100, 32), (64, 33), (128, 129), (128, 224), (60, 225), (128, 257),
                                   (1, 70), (4, 64), (5, 300), (100, 65), (127, 129), (128, 1000), (255, 63), (256, 64),
                                   (257, 600), (1023, 300), (1024, 257), (1025, 100), (8191, 40), (8192, 40)])
@pytest.mark.parametrize("act", ["Relu", "Softmax"])
def test_forward_over_entry_counts(kh, orc, dim, n, act):
    rng = np.random.default_rng(dim + n)
    layer, planes, W, b = slide_pair(kh, orc, dim, n, 3, 8, 64, FIFO, "Vanilla", 0, 2, act, rng)
    X = rows_of(rng, dim)
    check_slide(orc, layer, planes, W, b, X, layer.forward_batch(X), act == "Relu")


@pytest.mark.parametrize("act", ["Relu", "Softmax"])
def test_sparse_forward_over_entry_counts(kh, orc, act):
    from klearu_amd.lsh import SparseVector
    rng = np.random.default_rng(5)
    dim = 6000
    layer, planes, W, b = slide_pair(kh, orc, dim, 200, 3, 8, 64, FIFO, "Vanilla", 0, 2, act, rng)
    X = np.zeros((9, dim), np.float32)
    for x, c in zip(X, (0, 1, 16, 31, 32, 33, 4095, 4096, 4097)):
        x[rng.choice(dim, c, replace=False)] = rng.normal(0, 1, c)
    check_slide(orc, layer, planes, W, b, X, layer.forward_sparse_batch([SparseVector.from_dense(x) for x in X]),
                act == "Relu")
