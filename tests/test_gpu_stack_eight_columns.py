"""Products of up to 8 rows over up to 2048 columns, eight columns a workgroup (csrc/stack_ops.hip `stk_gemm_mfma_eight_kernel`): the bits of the tiles of 16
columns, which the same rows take among nine, and float64, at edges of columns, K-steps and waves, with rows gathered and scattered, a bias and a cap.

float32 sums of K products: 2e-6 of the result's norm, as for the other forms."""
import numpy as np
import pytest

from tests import stack_oracle as so
from tests.test_gpu_stack import BF16, check, empty, raw, rel, to_dev
from vllm_rs_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 3, 8])
@pytest.mark.parametrize("N,K", [(16, 32), (8, 8), (40, 72), (1001, 264), (2048, 2048), (2048, 520), (2041, 4104), (2049, 264), (1000, 8192)])
def test_eight_columns_a_workgroup(M, N, K):
    L = _lib.load()
    r = np.random.default_rng(M + N + K)
    a = so.bf16_round(r.standard_normal((9, K)).astype(np.float32))
    w = so.bf16_round((r.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32))
    ad, wd = to_dev(a, BF16), to_dev(w, BF16)

    def run(m, f32=1, rows=None, places=None):
        out = empty(10 * N * 4).fill_bytes(0)
        f = lambda v: None if v is None else raw(np.array(v), np.int32).ptr
        L.vra_stack_op_gemm(ad.ptr, K, wd.ptr, 0, out.ptr, N, f32, m, N, K, 0.5, None, 0, f(rows), None, f(places), 0, 0.0, BF16, 0)
        check()
        return out.numpy(np.uint32 if f32 else np.uint16, (10, N))

    nine = run(9)
    got = run(M)
    assert (got[:M] == nine[:M]).all() and (got[M:] == 0).all()
    assert rel(got[:M].view(np.float32), 0.5 * (a[:M].astype(np.float64) @ w.astype(np.float64).T)) < 2e-6
    assert (run(M, f32=0)[:M] == run(9, f32=0)[:M]).all()
    pick = [(5 * i + 8) % 9 for i in range(M)]
    if M > 1:
        pick[1] = -1
    moved = run(M, rows=pick, places=[9 - i for i in range(M)])
    for i in range(M):
        assert (moved[9 - i] == (nine[pick[i]] if pick[i] >= 0 else 0)).all()
