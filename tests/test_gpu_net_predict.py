"""GPU parity: Network.predict_batch / predict_sparse, whose examples run as rows of
one batch, against the oracle's one-example forward.

Bar: bit-exact, as training and prediction are (every f32 operation is the
reference's, in its order).
"""
import numpy as np
import pytest
import torch

from test_gpu_slide_train import build, spec

pytestmark = pytest.mark.gpu

F = np.float32


def inputs(rng, n, dim, density=0.3):
    return (rng.random((n, dim)) * (rng.random((n, dim)) < density)).astype(F)


@pytest.mark.parametrize("dim,hidden,out,batch,samp,act", [
    (96, 160, 120, 1, "TopK", "Relu"),          # one row
    (784, 256, 33, 129, "TopK", "Relu"),        # odd counts, several waves of active neurons
    (2500, 300, 64, 5, "Vanilla", "Sigmoid"),   # wider than the per-row hash kernel: the staged lists hash
    (64, 70, 40, 17, "Threshold", "Identity"),
])
def test_predict_rows_match_oracle(kh, orc, dim, hidden, out, batch, samp, act):
    from klearu_amd.lsh import SparseVector
    rng = np.random.default_rng(dim + batch)
    specs = [spec(rng, dim, hidden, act, sampling=samp, top_k=max(1, hidden // 4), k=5, L=8, cap=24, seed=3),
             spec(rng, hidden, out, "Softmax", top_k=max(1, out // 2), k=5, L=8, cap=24, seed=4)]
    net, layers, onet = build(orc, specs)
    X = inputs(rng, batch, dim)
    X[-1] = 0.0                                 # nothing but zeros
    got = net.predict_batch(X).cpu().numpy()
    sparse = net.predict_sparse([SparseVector.from_dense(x) for x in X]).cpu().numpy()
    for i in range(batch):
        np.testing.assert_array_equal(got[i], onet.predict(X[i]))
        np.testing.assert_array_equal(sparse[i], got[i])


def test_predict_more_rows_than_the_scratch_holds(kh, orc):
    """200000 outputs: about 50 rows at a time; 70 rows, and one row again."""
    rng = np.random.default_rng(77)
    specs = [spec(rng, 20, 16, "Relu", k=2, L=4, cap=16, seed=5),
             spec(rng, 16, 200000, "Softmax", top_k=50, k=8, L=4, cap=16, seed=6)]
    net, layers, onet = build(orc, specs)
    X = inputs(rng, 70, 20, 0.6)
    got = net.predict_batch(X).cpu().numpy()
    for i in (0, 1, 40, 60, 69):
        np.testing.assert_array_equal(got[i], onet.predict(X[i]))
    np.testing.assert_array_equal(net.predict_batch(X[60:61]).cpu().numpy()[0], got[60])


@pytest.mark.parametrize("family", ["WtaHash", "DwtaHash", "MinHash"])
def test_predict_rank_families_hash_the_lists(kh, family):
    """Rank-based families hash the staged lists (DWTA's sparse form differs from its dense one)."""
    from klearu_amd.lsh import LshConfig, SparseVector
    from klearu_amd.slide import Layer, LayerConfig, Network
    rng = np.random.default_rng(8)
    cfg = LayerConfig(60, 90, "Relu", LshConfig(hash_function=family, num_tables=6, num_hashes=4, bucket_capacity=16),
                      "Vanilla", 2, 0)
    layer = Layer(cfg, rng.standard_normal((90, 60)).astype(F), np.zeros(90, F), 9)
    net = Network([layer])
    X = inputs(rng, 7, 60)
    got = net.predict_batch(X).cpu().numpy()
    off, ids, _, act = (t.cpu().numpy() for t in layer.forward_sparse_batch([SparseVector.from_dense(x) for x in X]))
    want = np.zeros((7, 90), F)
    for i in range(7):
        want[i, ids[off[i]:off[i + 1]]] = act[off[i]:off[i + 1]]
    np.testing.assert_array_equal(got, want)


def test_predict_captured_before_its_rows_fit(kh, orc):
    """A larger batch than any before is captured all the same, and its replays are the eager
    results."""
    rng = np.random.default_rng(12)
    specs = [spec(rng, 40, 50, "Relu", top_k=20, k=4, L=5, cap=16, seed=7),
             spec(rng, 50, 30, "Softmax", top_k=10, k=4, L=5, cap=16, seed=8)]
    net, layers, onet = build(orc, specs)
    X = torch.from_numpy(inputs(rng, 6, 40)).cuda()
    net.predict_batch(X[:1])
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        out = net.predict_batch(X)
    for _ in range(3):
        X.copy_(torch.from_numpy(inputs(rng, 6, 40)).cuda())
        g.replay()
        torch.cuda.synchronize()
        got = out.cpu().numpy()
        for i, x in enumerate(X.cpu().numpy()):
            np.testing.assert_array_equal(got[i], onet.predict(x))
        np.testing.assert_array_equal(net.predict_batch(X).cpu().numpy(), got)


@pytest.mark.parametrize("streams,threads", [(2, 1), (3, 3), (1, 3)])
def test_predictions_of_one_network_side_by_side(kh, orc, streams, threads):
    """Predictions do not mutate: several streams, and host threads sharing one, each get the
    outputs of their own inputs."""
    import threading
    from klearu_amd.lsh import SparseVector
    rng = np.random.default_rng(31)
    specs = [spec(rng, 300, 400, "Relu", top_k=100, k=5, L=8, cap=24, seed=9),
             spec(rng, 400, 200, "Softmax", top_k=60, k=5, L=8, cap=24, seed=10)]
    net, layers, onet = build(orc, specs)
    n = max(streams, threads)
    Xs = [inputs(rng, 40 + 30 * j, 300) for j in range(n)]
    want = [net.predict_batch(X).cpu().numpy() for X in Xs]
    for j in range(n):
        np.testing.assert_array_equal(want[j][0], onet.predict(Xs[j][0]))
    dev = [torch.from_numpy(X).cuda() for X in Xs]
    sv = [[SparseVector.from_dense(x) for x in X[:20]] for X in Xs]
    st = [torch.cuda.Stream() for _ in range(streams)]
    outs = [[] for _ in range(n)]
    torch.cuda.synchronize()

    def work(j, reps):
        for _ in range(reps):
            outs[j].append(net.predict_batch(dev[j], stream=st[j % streams]))
    if threads == 1:
        for _ in range(12):
            for j in range(n):
                work(j, 1)
                outs[j].append(net.predict_sparse(sv[j], stream=st[j % streams]))
    else:
        ts = [threading.Thread(target=work, args=(j, 12)) for j in range(n)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
    torch.cuda.synchronize()
    for j in range(n):
        assert len(outs[j]) >= 12
        for o in outs[j]:
            np.testing.assert_array_equal(o.cpu().numpy(), want[j][:o.shape[0]])
