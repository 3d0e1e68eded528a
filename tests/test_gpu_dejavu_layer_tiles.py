"""GPU parity: the klearu-dejavu layer's kernels at the edges of their tiles (16 rows and
4 tokens per block, 128 steps per chunk, four chunks in flight) and the thread-per-output
forms, which short sums and many outputs take, vs the oracle.  Bar: bit-exact."""
import numpy as np
import pytest
import torch

from test_gpu_dejavu_layer import bits, xavier

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("in_f,out_f,batch", [
    (1, 1, 1), (3, 17, 2), (4, 15, 5), (127, 16, 3), (128, 33, 4), (129, 31, 6), (512, 20, 1), (516, 18, 2),
    (640, 48, 7), (20, 1024, 96), (37, 1100, 90), (16, 6200, 64), (33, 99000, 1), (48, 33000, 3),
    (96, 65, 3), (97, 17, 5), (100, 2049, 16), (100, 2048, 16), (140, 8, 2049), (600, 3100, 32)])
def test_linear_tile_edges(kh, orc, in_f, out_f, batch):
    from klearu_amd.dejavu_transformer import Linear
    rng = np.random.default_rng(in_f * 7 + out_f + batch)
    w, b = xavier(rng, out_f, in_f), rng.normal(0, 0.1, out_f).astype(np.float32)
    x = rng.standard_normal((batch, in_f)).astype(np.float32)
    x[0, ::3] = 0.0
    # a base 4 bytes past a 16-byte boundary: no vector loads of the inputs
    pad = torch.zeros(batch * in_f + 1, device="cuda")
    pad[1:] = torch.from_numpy(x).reshape(-1)
    lin = Linear(w, b)
    idx = rng.integers(0, out_f, 19)
    for xd in (torch.from_numpy(x).cuda(), pad[1:].view(batch, in_f)):
        y, ys = lin.forward(xd).cpu().numpy(), lin.forward_sparse(xd, idx).cpu().numpy()
        for r in sorted({0, batch // 2, batch - 1}):
            ref = orc.dejavu_linear_forward(w, b, x[r])
            np.testing.assert_array_equal(bits(y[r]), bits(ref))
            np.testing.assert_array_equal(bits(ys[r]), bits(ref[idx]))


@pytest.mark.parametrize("H,I,n,batch", [(1, 1, 1, 1), (17, 40, 9, 3), (64, 300, 129, 5), (130, 90, 8, 2), (20, 700, 640, 4),
                                         (97, 40, 9, 3), (132, 300, 129, 5), (200, 80, 32, 160), (200, 80, 33, 160),
                                         (200, 80, 17, 160), (100, 120, 100, 170), (100, 120, 120, 500),
                                         (300, 60, 31, 1025), (64, 40, 1, 2050)])
def test_sparse_mlp_tile_edges(kh, orc, H, I, n, batch):
    """Non-finite weights of a neuron whose activation is zero add nothing."""
    from klearu_amd.dejavu_transformer import Linear, SparseMlp
    rng = np.random.default_rng(H + I + n)
    wg, wu, wd = xavier(rng, I, H), xavier(rng, I, H), xavier(rng, H, I)
    bg, bu, bd = (rng.normal(0, 0.05, m).astype(np.float32) for m in (I, I, H))
    wu[0], bu[0] = 0.0, 0.0
    wd[:, 0] = np.inf
    x = rng.standard_normal((batch, H)).astype(np.float32)
    sel = rng.choice(I, n, replace=False)
    sel[0] = 0
    y = SparseMlp(H, I).forward(torch.from_numpy(x).cuda(), Linear(wg, bg), Linear(wu, bu), Linear(wd, bd), sel)
    for r in range(batch) if batch < 8 else sorted({0, 1, 2, batch // 2, batch - 2, batch - 1}):
        ref = orc.dejavu_sparse_mlp_forward(wg, bg, wu, bu, wd, bd, x[r], sel)
        np.testing.assert_array_equal(bits(y[r].cpu().numpy()), bits(ref))


@pytest.mark.parametrize("H,nh,hd,batch", [(24, 3, 1, 2), (40, 2, 63, 1), (32, 2, 65, 5), (16, 1, 200, 3)])
def test_sparse_attention_head_dims(kh, orc, H, nh, hd, batch):
    from klearu_amd.dejavu_transformer import Linear, SparseAttention
    rng = np.random.default_rng(H + hd)
    ws = [xavier(rng, nh * hd, H) for _ in range(3)] + [xavier(rng, H, nh * hd)]
    bs = [rng.normal(0, 0.05, w.shape[0]).astype(np.float32) for w in ws]
    x = rng.standard_normal((batch, H)).astype(np.float32)
    heads = [nh - 1]
    y = SparseAttention(H, nh, hd).forward(torch.from_numpy(x).cuda(), *(Linear(w, b) for w, b in zip(ws, bs)), heads)
    args = [a for pair in zip(ws, bs) for a in pair]
    for r in range(batch):
        ref = orc.dejavu_sparse_attention_forward(*args, nh, hd, x[r], heads)
        np.testing.assert_array_equal(bits(y[r].cpu().numpy()), bits(ref))


@pytest.mark.parametrize("n", [960, 961])
def test_index_list_in_the_launch_and_copied(kh, orc, n):
    from klearu_amd.dejavu_transformer import Linear
    rng = np.random.default_rng(n)
    w, b = xavier(rng, 500, 12), rng.normal(0, 0.1, 500).astype(np.float32)
    x = rng.standard_normal(12).astype(np.float32)
    idx = rng.integers(0, 500, n)
    y = Linear(w, b).forward_sparse(x, idx).cpu().numpy()
    np.testing.assert_array_equal(bits(y), bits(orc.dejavu_linear_forward(w, b, x)[idx]))


def test_creating_a_linear_leaves_other_streams_running(kh):
    """The upload is waited for on its own stream; work queued on another goes on meanwhile."""
    from klearu_amd.dejavu_transformer import Linear
    side = torch.cuda.Stream()
    a = torch.randn(4096, 4096, device="cuda")
    Linear(np.ones((64, 64), np.float32))
    torch.cuda.synchronize()
    done = torch.cuda.Event()
    with torch.cuda.stream(side):
        for _ in range(200):
            a = torch.tanh(a @ a)
        done.record()
    lin = Linear(np.ones((64, 64), np.float32))
    assert not done.query()
    torch.cuda.synchronize()
    assert float(lin.forward(np.ones(64, np.float32))[3]) == 64.0
