"""CSR rows written by the forward kernels: 4096 rows (the most whose offsets the kernels
sum) against 4097 (packed by another launch); outputs left out; and outputs too small,
where the call fails and every entry that has room is still the one of the full call."""
import numpy as np
import pytest
import torch

from test_gpu_lsh_slide import FIFO, slide_pair

pytestmark = pytest.mark.gpu


def forward(layer, X, cap, pre=True, act=True):
    from klearu_amd import _lib
    from klearu_amd._dev import ptr
    B = X.shape[0]
    off = torch.zeros(B + 1, dtype=torch.int64, device="cuda")
    ids = torch.full((cap,), -1, dtype=torch.int32, device="cuda")
    z = [torch.full((cap,), -1.0, device="cuda") for _ in range(2)]
    rc = _lib.load().kh_slide_layer_forward(layer._h, ptr(X), B, ptr(off), ptr(ids), ptr(z[0]) if pre else None,
                                           ptr(z[1]) if act else None, cap, None)
    torch.cuda.synchronize()
    return rc, off.cpu(), [t.cpu() for t in (ids, *z)]


@pytest.mark.parametrize("dim,n,act", [(20, 30, "Relu"), (20, 30, "Softmax"), (21, 30, "Softmax"), (200, 700, "Tanh")])
def test_rows_in_place(kh, orc, dim, n, act):
    rng = np.random.default_rng(dim + n)
    layer, *_ = slide_pair(kh, orc, dim, n, 3, 4, 8, FIFO, "Vanilla", 0, 2, act, rng)
    X = torch.from_numpy(rng.normal(0, 1, (4097, dim)).astype(np.float32)).cuda()
    cap = 4097 * n
    rc, off, full = forward(layer, X, cap)
    assert rc == 0
    rc, off2, got = forward(layer, X[:4096], cap)
    assert rc == 0
    m = int(off2[-1])
    assert torch.equal(off2, off[:4097])
    for a, b in zip(got, full):
        assert torch.equal(a[:m], b[:m]) and bool((a[m:] == -1).all())
    rows = X[:5].contiguous()
    m = int(off[5])
    for keep in ((True, False), (False, True)):
        rc, o, got = forward(layer, rows, cap, *keep)
        assert rc == 0 and torch.equal(o, off[:6])
        for a, b, k in zip(got, full, (True, *keep)):
            assert torch.equal(a[:m], b[:m]) if k else bool((a == -1).all())
    for short in (1, m - int(off[4]), m - 1):     # nothing but the last entry, the last row, all but one
        rc, o, got = forward(layer, rows, m - short)
        assert rc != 0 and torch.equal(o, off[:6])
        for a, b in zip(got, full):
            assert torch.equal(a, b[:m - short])
