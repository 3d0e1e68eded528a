"""Queries over buckets whose fill meets the lanes (sixteen or more) and the two or eight entries a
lane: one entry to several rounds, empty buckets beside full ones, few and many tables, one
row (1024 threads) and many, ids for the direct, the bitmap and the sorting path."""
import numpy as np
import pytest
import torch

from test_gpu_lsh_slide import FIFO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [1, 40])
@pytest.mark.parametrize("L,fill,bound", [(1, 5000, 12000), (1, 8192, 300000), (2, 4096, 300000), (3, 1000, 12000),
                                          (8, 700, 300000), (9, 700, 12000), (16, 400, 300000), (32, 200, 12000)])
def test_query_few_large_buckets(kh, rows, L, fill, bound):
    """Up to a whole block of lanes walks one bucket."""
    test_query_at_bucket_fills(kh, rows, L, fill, bound)


@pytest.mark.parametrize("rows", [1, 40])
@pytest.mark.parametrize("L,fill", [(1, 1), (3, 15), (5, 16), (64, 17), (65, 32), (50, 33), (2, 127), (33, 128), (7, 129), (4, 300)])
@pytest.mark.parametrize("bound", [700, 300000, 1 << 31])
def test_query_at_bucket_fills(kh, rows, L, fill, bound):
    from klearu_amd.lsh import HashFamily, LshIndex
    rng = np.random.default_rng(L * 1000 + fill)
    # planes of zeros: every query's code is 3 in every table
    idx = LshIndex(HashFamily.from_planes(np.zeros((L, 2, 4), np.int8)), FIFO, fill)
    n = 2 * fill + 3
    ids = rng.choice(bound, n, replace=False) if n <= bound < 1 << 20 else np.unique(rng.integers(0, bound, n))
    codes = np.where(rng.uniform(size=(len(ids), L)) < rng.choice([0.0, 0.3, 1.0], L), 3, 0)
    codes[0] = 3
    idx.insert_codes(ids.astype(np.uint32), codes.astype(np.uint32))
    data, ln, _ = idx.buckets()
    want = np.unique(np.concatenate([data[t, 3, :ln[t, 3]] for t in range(L)]), return_counts=True)
    assert len(want[0])
    X = torch.ones(rows, 4, device="cuda")
    for counts in (True, False):
        off, qi, qc = idx.query_batch(X, counts=counts)
        off, qi = off.cpu().numpy(), qi.cpu().numpy().view(np.uint32)
        for r in range(rows):
            np.testing.assert_array_equal(qi[off[r]:off[r + 1]], want[0])
            if counts:
                np.testing.assert_array_equal(qc[off[r]:off[r + 1]].cpu().numpy(), want[1])
