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
    x[0, :2], x[M // 2, -1], w[0, 1, 0] = (3e38, 1e-41), 1e-30, 2e38  # overflow, underflow, denormals
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
