"""Products of up to 8 rows over up to 2048 columns, eight columns a workgroup (csrc/stack_ops.hip `stk_gemm_mfma_eight_kernel`): the bits of the tiles of 16
columns, which the same rows take among nine, and float64, at edges of columns, K-steps and waves: rows gathered and scattered, a bias, activations and a cap,
and batches with strides of their own.

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


# (2048 and 8200 channels: two rounds of loads a wave and more, the last one short; 264: one step of two waves only)
@pytest.mark.parametrize("M", [1, 3, 8])
@pytest.mark.parametrize("N,K", [(40, 264), (1001, 2048), (2047, 8200)])
def test_bias_activations_and_cap(M, N, K):
    L = _lib.load()
    r = np.random.default_rng(M + N + K)
    a = so.bf16_round(r.standard_normal((9, K)).astype(np.float32))
    w = so.bf16_round((r.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32))
    bias = r.standard_normal(N).astype(np.float32)
    ad, wd, bd = to_dev(a, BF16), to_dev(w, BF16), raw(bias, np.float32)
    z = 1.5 * (a.astype(np.float64) @ w.astype(np.float64).T)

    def run(m, b, epi, act, cap, f32=1):
        out = empty(9 * N * 4).fill_bytes(0)
        L.vra_stack_op_gemm_post(ad.ptr, K, wd.ptr, 0, out.ptr, N, f32, m, N, K, 1.5, bd.ptr if b else None, None, 0, None, None, epi, act, cap, BF16, 0)
        check()
        return out.numpy(np.uint32 if f32 else np.uint16, (9, N))

    for b, epi, act, cap, fn in [(1, 0, 0, 0.0, lambda v: v), (1, 0, 0, 2.5, lambda v: 2.5 * np.tanh(v / 2.5)), (0, 0, 0, 0.5, lambda v: 0.5 * np.tanh(v / 0.5)),
                                 (0, 2, 3, 0.0, None), (1, 2, 4, 0.0, lambda v: np.maximum(v, 0.0) ** 2), (1, 2, 5, 0.0, np.tanh), (1, 2, 6, 1.5, None)]:
        got, nine = run(M, b, epi, act, cap), run(9, b, epi, act, cap)
        assert (got[:M] == nine[:M]).all() and (got[M:] == 0).all(), (b, epi, act, cap)
        assert (run(M, b, epi, act, cap, 0)[:M] == run(9, b, epi, act, cap, 0)[:M]).all()
        if fn is not None:
            assert rel(got[:M].view(np.float32), fn(z[:M] + (bias if b else 0.0))) < 4e-6, (b, epi, act, cap)  # (the sum's 2e-6, at most doubled by the square)


@pytest.mark.parametrize("M", [1, 8])
@pytest.mark.parametrize("nb,N,K,os_", [(3, 520, 2056, 528), (16, 128, 264, 128), (5, 41, 8200, 48)])
def test_batches(M, nb, N, K, os_):
    """one product a batch: columns z * K .. of the rows, weights and outputs of its own, places between the outputs left alone"""
    L = _lib.load()
    r = np.random.default_rng(M + N + K)
    a = so.bf16_round(r.standard_normal((9, nb * K)).astype(np.float32))
    w = so.bf16_round((r.standard_normal((nb, N, K)) / np.sqrt(K)).astype(np.float32))
    ad, wd = to_dev(a, BF16), to_dev(w, BF16)

    def run(m):
        out = empty(9 * nb * os_ * 4).fill_bytes(0)
        L.vra_stack_op_gemm_ex(ad.ptr, nb * K, wd.ptr, out.ptr, nb * os_, 1, m, N, K, 1.0, None, 0, 0, nb, K, N * K, os_, BF16, 0)
        check()
        return out.numpy(np.uint32, (9, nb, os_))

    got, nine = run(M), run(9)
    assert (got[:M] == nine[:M]).all() and (got[M:] == 0).all() and (got[:, :, N:] == 0).all()
    for z in range(nb):
        assert rel(got[:M, z, :N].view(np.float32), a[:M, z * K:(z + 1) * K].astype(np.float64) @ w[z].astype(np.float64).T) < 2e-6
