"""The f32 matrix products of a layer stack on the matrix units (csrc/stack_ops.hip): the bits of the form without them, which rows off 16 bytes take."""
import numpy as np
import pytest

from tests.util import F32, rng
from vllm_rs_amd import _lib, ops

pytestmark = pytest.mark.gpu


# rows around 16, 32 and 64, columns that end inside a tile of 16 and take tiles of 16 x 16, (130 rows:) 32 x 16 and 32 x 32,
# K of less than a block of 16, off it, of less and more blocks than are read ahead
@pytest.mark.parametrize("M", [1, 16, 17, 33, 65, 130])
@pytest.mark.parametrize("N", [5, 300, 1500, 3001])
@pytest.mark.parametrize("K", [4, 36, 272, 520])
@pytest.mark.parametrize("form", ["plain", "rows", "groups"])
def test_f32_product(form, M, N, K):
    L = _lib.load()
    r = rng(M * 7 + N + K)
    g = 64 if M > 32 else 16
    if form == "groups":
        M = -(-M // g) * g
    x, w = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((3, N, K)).astype(np.float32)
    x[0, :2], w[0, 1, 0] = (3e38, 1e-41), 2e38  # overflow
    gid = r.integers(-1, 3, max(M // g, 1)).astype(np.int32) if form == "groups" else None
    src = r.permutation(M).astype(np.int32) if form == "rows" else None
    dst = r.permutation(M + 1)[:M].astype(np.int32) if form == "rows" else None
    if src is not None and M > 1:
        src[-1], dst[0] = -1, -1  # a row without an input, one without an output
    sc = r.standard_normal(M).astype(np.float32) if form != "plain" else None
    dev = lambda v: ops.dev(v.view(np.uint32)) if v is not None else None
    p = lambda b: b.ptr if b else None
    gd, sd, dd, scd, wd = dev(gid), dev(src), dev(dst), dev(sc), ops.dev(w)

    def run(lda):
        xd = ops.dev(np.ascontiguousarray(np.pad(x, ((0, 0), (0, lda - K)))))
        out = ops.DevBuf((M + 1) * N * 4).fill_bytes(0)
        L.vra_stack_op_gemm(xd.ptr, lda, wd.ptr, N * K if form == "groups" else 0, out.ptr, N, 1, M, N, K, 0.5, p(gd), g, p(sd), p(scd), p(dd), 0, 0.0, F32, 0)
        ops.check_error()
        return out.numpy(np.float32, (M + 1, N))
    got, want = run(K + 4), run(K + 1)
    assert np.array_equal(got, want, equal_nan=True) and (form == "groups" or got.any())  # (all of a group may be holes)


# sums that stay below the least normal number: denormal operands, denormal products of normal ones, normal products that cancel
@pytest.mark.parametrize("M,N", [(3, 40), (130, 300), (130, 3001)])
@pytest.mark.parametrize("K", [4, 36, 272, 520])
def test_f32_product_of_tiny_numbers(K, M, N):
    L = _lib.load()
    r = rng(K + M + N)
    x, w = r.standard_normal((M, K)).astype(np.float32), r.standard_normal((N, K)).astype(np.float32)
    x[0::3] *= np.float32(1e-41)
    x[1::3] *= np.float32(1e-25)
    x[2::3] = np.float32(1.5e-38) * (1 - 2 * (np.arange(K) % 2)) * (1 + np.arange(K) % 2 * np.float32(2.0 ** -10))
    w[0::2] *= np.float32(1e-18)  # (with rows 1, 4, ..: 1e-43; with the others underflow to zero)
    w[1::4] = 1.0
    wd = ops.dev(w)

    def run(lda):
        xd = ops.dev(np.ascontiguousarray(np.pad(x, ((0, 0), (0, lda - K)))))
        out = ops.DevBuf(M * N * 4).fill_bytes(0xEE)
        L.vra_stack_op_gemm(xd.ptr, lda, wd.ptr, 0, out.ptr, N, 1, M, N, K, 1.0, None, 0, None, None, None, 0, 0.0, F32, 0)
        ops.check_error()
        return out.numpy(np.float32, (M, N))
    got, want = run(K + 4), run(K + 1)
    assert np.array_equal(got.view(np.uint32), want.view(np.uint32))
    tiny = np.float64(2.0 ** -126)
    exact = x.astype(np.float64) @ w.astype(np.float64).T
    # (an addition is exact below 2 ** -126; products round to the spacing of denormals, here once a product and once more where a fused step does not)
    for rows, cols in ((slice(0, None, 3), slice(1, None, 4)), (slice(1, None, 3), slice(0, None, 2)), (slice(2, None, 3), slice(1, None, 4))):
        e, g = exact[rows, cols], got[rows, cols].astype(np.float64)
        assert np.abs(e).max() < tiny and np.count_nonzero(g) > g.size // 2
        assert np.abs(g - e).max() <= K * 2.0 ** -149
