"""GPU parity: the accel kernels at the edges of their tiles and at unaligned addresses, vs
the oracle.  Bar: bit-exact."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

F = np.float32


def bits(a):
    return np.asarray(a, F).view(np.uint32)


def at_offset(a, off):
    """A device copy of `a` that starts `off` elements past an aligned address."""
    t = torch.from_numpy(np.ascontiguousarray(a))
    buf = torch.zeros(t.numel() + off, dtype=t.dtype, device="cuda")
    buf[off:] = t.reshape(-1).cuda()
    return buf[off:].view(t.shape)


@pytest.mark.parametrize("n", [1, 15, 16, 24, 255, 256, 257, 511, 512, 528, 776, 1027, 4096])
@pytest.mark.parametrize("rows", [1, 17])
def test_dense_dot_groups(kh, orc, rows, n):
    from klearu_amd.accel import dense_dot_dense_simd
    rng = np.random.default_rng(n + rows)
    A, b = rng.standard_normal((rows, n)).astype(F), rng.standard_normal(n).astype(F)
    got = dense_dot_dense_simd(at_offset(A, 1), at_offset(b, 3)).cpu().numpy()
    np.testing.assert_array_equal(bits(got), bits([orc.dense_dot(a, b) for a in A]))


@pytest.mark.parametrize("nnz", [1, 7, 8, 2047, 2048, 2049, 2056, 4096, 4103, 9000])
def test_sparse_dot_tiles(kh, orc, nnz):
    from klearu_amd.accel import sparse_dot_dense_simd
    rng = np.random.default_rng(nnz)
    dense = rng.standard_normal(10000).astype(F)
    idx, val = np.sort(rng.choice(10000, nnz, replace=False)).astype(np.uint32), rng.standard_normal(nnz).astype(F)
    got = float(sparse_dot_dense_simd(idx, val, torch.from_numpy(dense).cuda()))
    assert F(got).tobytes() == orc.sparse_dot_dense(idx, val, dense).tobytes()


@pytest.mark.parametrize("n,span", [(1, 5), (1023, 1 << 20), (1024, 1024), (1025, 900), (3000, 1), (2500, 100000)])
def test_scatter_add_chunks(kh, orc, n, span):
    """Distinct, colliding and all-equal indices; an index repeated across chunks."""
    from klearu_amd.accel import scatter_add_simd
    rng = np.random.default_rng(n + span)
    idx = (rng.integers(0, span, n) if n != 1024 else rng.permutation(1024)).astype(np.uint32)
    idx[-1] = idx[0]
    val, d0 = rng.standard_normal(n).astype(F), rng.standard_normal(span).astype(F)
    got = scatter_add_simd(idx, val, torch.from_numpy(d0).cuda(), -1.25).cpu().numpy()
    np.testing.assert_array_equal(bits(got), bits(orc.scatter_add(idx, val, d0, -1.25)))


@pytest.mark.parametrize("n", [1, 7, 8, 9, 8191, 8192, 8200, 50003])
@pytest.mark.parametrize("off", [0, 1, 8])
def test_bf16_conversions(kh, orc, n, off):
    """Eight elements per access where both arrays are aligned; NaN, infinities, ties, denormals."""
    from klearu_amd._dev import ptr, stream_ptr
    from klearu_amd.accel import Bf16Weights
    rng = np.random.default_rng(n + off)
    x = rng.integers(0, 1 << 32, n, dtype=np.uint64).astype(np.uint32).view(F)
    w = Bf16Weights.from_f32(at_offset(x, off))
    ref = orc.bf16_from_f32(x)
    np.testing.assert_array_equal(w.data.cpu().numpy().view(np.uint16), ref)
    np.testing.assert_array_equal(bits(Bf16Weights(at_offset(ref.view(np.int16), off)).to_f32().cpu().numpy()),
                                  bits(orc.bf16_to_f32(ref)))
    v = orc.bf16_from_f32(rng.standard_normal(n).astype(F))
    d = (rng.standard_normal(n) * 0.01).astype(F)
    u = Bf16Weights(at_offset(v.view(np.int16), off))
    u.update_from_f32(at_offset(d, off))
    np.testing.assert_array_equal(u.data.cpu().numpy().view(np.uint16), orc.bf16_update_from_f32(v, d))


@pytest.mark.parametrize("rows", [1, 16, 19])
@pytest.mark.parametrize("n", [1, 3, 127, 128, 511, 512, 513, 2048, 2052, 5000])
def test_bf16_dot_rows(kh, orc, rows, n):
    from klearu_amd import _lib
    from klearu_amd._dev import ptr, stream_ptr
    from klearu_amd.accel import bf16_full_dot
    rng = np.random.default_rng(n * 3 + rows)
    w = orc.bf16_from_f32(rng.standard_normal((rows, n)).astype(F).reshape(-1)).reshape(rows, n)
    x = rng.standard_normal(n).astype(F)
    for off in (0, 1):
        wd, xd = at_offset(w.view(np.int16), off), at_offset(x, off)
        out = torch.empty(rows, dtype=torch.float32, device="cuda")
        _lib.call("kh_bf16_dot_f32", ptr(wd), rows, n, ptr(xd), n, ptr(out), stream_ptr())
        np.testing.assert_array_equal(bits(out.cpu().numpy()), bits([orc.bf16_dot_f32(r, x) for r in w]))
    xb = orc.bf16_from_f32(x)
    got = F(float(bf16_full_dot(at_offset(w[0].view(np.int16), 0), at_offset(xb.view(np.int16), 1))))
    assert got.tobytes() == orc.bf16_full_dot(w[0], xb).tobytes()


@pytest.mark.parametrize("rows,n,ldw", [(1, 16, 16), (1, 17, 17), (65, 0, 4), (64, 1, 3), (2, 16, 20), (2549, 17, 17),
                                        (2550, 17, 21), (3900, 26, 26), (3899, 26, 28)])
def test_bf16_dot_short_rows(kh, orc, rows, n, ldw):
    """Short rows take a thread each: one row to many, on both sides of the rule."""
    from klearu_amd import _lib
    from klearu_amd._dev import ptr, stream_ptr
    rng = np.random.default_rng(rows + n)
    w = orc.bf16_from_f32(rng.standard_normal(rows * ldw).astype(F)).reshape(rows, ldw)
    x = rng.standard_normal(max(n, 1)).astype(F)[:n]
    wd, xd = at_offset(w.view(np.int16), 1), at_offset(np.append(x, F(0)), 1)
    out = torch.full((rows,), 7.0, dtype=torch.float32, device="cuda")
    _lib.call("kh_bf16_dot_f32", ptr(wd), rows, ldw, ptr(xd), n, ptr(out), stream_ptr())
    want = [orc.bf16_dot_f32(np.ascontiguousarray(r[:n]), x) if n else F(-0.0) for r in w]
    np.testing.assert_array_equal(bits(out.cpu().numpy()), bits(want))
