"""Inserts by rank against the oracle's replay of each bucket, bit for bit: sizes around
a wave (64), a block's chunk (4096), the transposing of row-major codes (512) and the
tables too large to count (12 bits, sorted) and few inserts into many buckets (sorted); skewed codes, so that buckets overflow
within one chunk; a second call into buckets that hold entries, with fewer and with more
inserts than they keep."""
import numpy as np
import pytest

from test_gpu_lsh_slide import FIFO, RESERVOIR, assert_buckets_equal

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bt", [FIFO, RESERVOIR])
@pytest.mark.parametrize("k,L,cap,n1,n2", [(1, 1, 1, 1, 1), (3, 2, 6, 64, 65), (6, 33, 128, 511, 513),
                                           (9, 5, 7, 4095, 4097), (11, 3, 16, 12345, 700), (11, 70, 4, 1, 4096),
                                           (12, 2, 8, 5000, 900), (6, 10, 16, 256, 257), (5, 4, 16, 2048, 2049), (11, 256, 4, 509, 510)])
def test_inserts_by_rank_match_the_replay(kh, orc, bt, k, L, cap, n1, n2):
    from klearu_amd.lsh import LshIndex, SimHash
    rng = np.random.default_rng(k * 100 + n1)
    idx = LshIndex(SimHash(16, k, L, 5), bt, cap)
    ref = orc.LshIndex(L, k, cap, bt)
    for n in (n1, n2, 3):
        ids = rng.integers(0, 10 * n, n).astype(np.uint32)
        codes = (rng.integers(0, 1 << k, (n, L)) * (rng.uniform(size=(n, L)) < 0.7)).astype(np.uint32)
        idx.insert_codes(ids, codes)
        ref.insert_many(ids, codes)
        assert_buckets_equal(idx, ref)


@pytest.mark.parametrize("bt", [FIFO, RESERVOIR])
def test_inserts_of_more_than_256_chunks_worth(kh, orc, bt):
    """Above 256 x 4096 vectors a chunk grows: 2^20 + 1 is the first such size."""
    from klearu_amd.lsh import LshIndex, SimHash
    n = (1 << 20) + 1
    rng = np.random.default_rng(1)
    idx = LshIndex(SimHash(16, 4, 1, 5), bt, 32)
    ref = orc.LshIndex(1, 4, 32, bt)
    codes = rng.integers(0, 16, (n, 1)).astype(np.uint32)
    idx.insert_codes(np.arange(n, dtype=np.uint32), codes)
    ref.insert_many(np.arange(n, dtype=np.uint32), codes)
    assert_buckets_equal(idx, ref)
