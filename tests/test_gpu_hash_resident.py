"""GPU parity: hashing of large dense batches with the planes resident in LDS (up to 128
dimensions, planes that fit), at the edges of its tiles: k steps of 32 dimensions, 16-plane
tiles, 16-row tiles, more rows than one pass of the grid, rows of inf / NaN, a queue of
undecided signs that overflows; and of wider batches, whose planes are read again, with rows
that allow whole pieces, none, and too many values for either.  Bar: bit-exact codes."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,k,L,batch", [
    (1, 1, 1, 1024), (31, 3, 7, 1025), (32, 24, 3, 1030), (33, 9, 50, 1040), (64, 5, 13, 1999), (96, 6, 50, 1500),
    (100, 7, 37, 1100), (127, 9, 50, 1031), (128, 9, 50, 70001), (128, 1, 17, 1024),
    (4, 9, 50, 1025), (36, 9, 50, 1300), (65, 9, 50, 1100), (130, 5, 20, 1040), (204, 5, 20, 1040), (512, 4, 11, 1030),
    (511, 4, 11, 1030), (513, 4, 11, 1030), (2001, 2, 9, 1025)])
def test_resident_codes(kh, orc, dim, k, L, batch):
    from klearu_amd.lsh import HashFamily
    rng = np.random.default_rng(dim * 100 + k)
    planes = rng.choice(np.array([-1, 0, 0, 0, 0, 1], np.int8), (L, k, dim))
    x = (rng.standard_normal((batch, dim)) * 0.01).astype(np.float32)
    x[1] = 0.0                                     # every sign a tie: the queue overflows
    x[2, dim // 2] = np.inf
    x[3, 0] = np.nan
    x[4] = rng.choice(np.array([-1, 1], np.float32), dim)           # exact cancellations
    x[5] *= 1e-38
    x[6] *= 1e37
    fam = HashFamily.from_planes(planes)
    pad = torch.zeros(batch * dim + 1, device="cuda")
    pad[1:] = torch.from_numpy(x).reshape(-1)
    rows = np.unique(np.concatenate([np.arange(40), rng.integers(0, batch, 200), np.arange(batch - 20, batch)]))
    want = orc.hash_dense_batch(planes, x[rows])
    for xd in (torch.from_numpy(x).cuda(), pad[1:].view(batch, dim)):
        got = fam.hash_dense_batch(xd).cpu().numpy().view(np.uint32)
        np.testing.assert_array_equal(got[rows], want)
