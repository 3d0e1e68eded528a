"""load_cache_dev against the loaded arrays, bit for bit: one row, a few blocks per head
and more than one step per block (5003 rows of two heads, 256 wide); sources off a
16-byte line; BF16 rows, and rows in which only the first or the last value is none."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("kv", [0, 1])
@pytest.mark.parametrize("nkv,length,dim", [(1, 1, 64), (3, 37, 128), (2, 5003, 256), (64, 301, 64)])
@pytest.mark.parametrize("shift", [0, 1])
@pytest.mark.parametrize("odd", [None, 0, -1])
def test_loaded_rows_read_back(kh, kv, nkv, length, dim, shift, odd):
    from klearu_amd.attention import SparseAttention
    w = np.zeros((nkv * dim, 64), np.uint16)
    a = SparseAttention(64, nkv, nkv, dim, w, w, w, np.zeros((64, nkv * dim), np.uint16), length + 2, 2, kv_dtype=kv)
    g = torch.Generator().manual_seed(length)
    n = nkv * length * dim
    rows = [torch.randn(n + shift, generator=g).to(torch.bfloat16).float()[shift:] for _ in range(2)]
    if odd is not None:
        rows[1][odd] = 1.0 + 2.0 ** -20
    dev = []
    for r in rows:
        buf = torch.zeros(n + shift, device="cuda")
        buf[shift:] = r.cuda()
        dev.append(buf[shift:].view(nkv, length, dim))
    a.load_cache_dev(1, *dev)
    torch.cuda.synchronize()
    assert a.current_len(1) == length and a.current_len(0) == 0
    for got, want in zip(a.read_cache(1, length), rows):
        np.testing.assert_array_equal(got, want.view(nkv, length, dim).numpy())
    a.load_cache_dev(1, dev[0][:, :0].contiguous(), dev[1][:, :0].contiguous())
    torch.cuda.synchronize()
    assert a.current_len(1) == 0
