"""Optimizer updates where the tiles of active weights (1024, over rows end to end) meet rows:
rows shorter than a tile, a tile's length and one more or less, several tiles; and staged
sparse examples in index order with repeated indices and zeros.  Bars as in test_gpu_slide_train."""
import numpy as np
import pytest

from test_gpu_slide_train import F, build, check_same, data, run_steps, spec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("optimizer,momentum", [("Sgd", 0.0), ("Sgd", 0.9), ("Adam", 0.9)])
@pytest.mark.parametrize("dim,n", [(3, 5), (341, 7), (1023, 9), (1024, 3), (1025, 33), (2500, 6)])
def test_update_tiles(kh, orc, dim, n, optimizer, momentum):
    rng = np.random.default_rng(dim + n)
    specs = [spec(rng, dim, n, "Relu", k=3, L=4, cap=64, seed=71), spec(rng, n, 5, "Softmax", k=3, L=4, cap=64, seed=72)]
    net, layers, onet = build(orc, specs, optimizer, momentum)
    X, labels = data(rng, 6, dim, 5)
    run_steps(net, layers, onet, X, labels, 0.01, 2, 3)


@pytest.mark.parametrize("nnz", [1, 2, 75, 1023, 1030])
def test_sorted_rows_with_repeats(kh, orc, nnz):
    from klearu_amd.lsh import SparseVector
    rng = np.random.default_rng(nnz)
    dim = 1500
    specs = [spec(rng, dim, 20, "Relu", k=3, L=4, cap=64, seed=73), spec(rng, 20, 6, "Softmax", k=3, L=4, cap=64, seed=74)]
    net, layers, onet = build(orc, specs, "Adam")
    vecs, X = [], np.zeros((4, dim), F)
    for r in range(4):
        idx = np.sort(rng.integers(0, dim, nnz)).astype(np.uint32)   # the later of equal indices wins
        val = rng.random(nnz).astype(F)
        val[::7] = 0.0
        for i, v in zip(idx, val):
            X[r, i] = v
        vecs.append(SparseVector(idx, val, dim))
    labels = [[int(rng.integers(0, 6))] for _ in range(4)]
    got, want = net.train_step_sparse(vecs, labels, 0.01), onet.train_step(X, labels, 0.01)
    assert got == pytest.approx(want, rel=1e-5)
    check_same(layers, onet, f"nnz {nnz}")
