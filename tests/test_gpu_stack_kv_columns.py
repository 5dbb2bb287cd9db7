"""The product whose key and value columns go to their cache rows (csrc/stack_ops.hip, StkGemmArgs::kv_slot): the bits of the plain product and the copy
behind it, in the forms of few rows (eight and sixteen columns a workgroup), on the prompt tiles, and where the copy is a launch of its own (widths
that are no 16-byte pieces, K off 64, rows off 16 bytes, float32).  Rows without a slot and cache rows that nobody names stay as they were."""
import numpy as np
import pytest

from tests import stack_oracle as so
from tests.test_gpu_stack import BF16, F32, check, empty, raw, rel, to_dev
from vllm_rs_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("M", [1, 8, 9, 17, 32, 33, 64, 130, 260])
@pytest.mark.parametrize("nq,nk,nv,K,pad,dt", [(256, 64, 64, 128, 0, BF16), (2048, 512, 512, 2048, 0, BF16), (192, 64, 128, 64, 8, BF16), (72, 24, 40, 192, 0, BF16), (1, 3, 5, 64, 0, BF16),
                                               (256, 64, 64, 72, 0, BF16), (256, 64, 64, 128, 4, BF16), (64, 32, 32, 64, 0, F32), (30, 10, 10, 30, 1, F32)])
def test_key_and_value_columns_go_to_their_rows(M, nq, nk, nv, K, pad, dt):
    L = _lib.load()
    r = np.random.default_rng(M + nq + K)
    N, ld, rows = nq + nk + nv, nq + nk + nv + pad, 300
    a = r.standard_normal((M, K + pad)).astype(np.float32)
    w = (r.standard_normal((N, K)) / np.sqrt(K)).astype(np.float32)
    if dt == BF16:
        a, w = so.bf16_round(a), so.bf16_round(w)
    slots = r.permutation(rows)[:M].astype(np.int64)
    slots[max(M // 2, 1)::7] = -1
    ad, wd, sd = to_dev(a, dt), to_dev(w, dt), raw(slots, np.int64)
    word = np.uint32 if dt == F32 else np.uint16
    es = 4 if dt == F32 else 2

    def run(fused):
        out, kc, vc = (empty(n * es).fill_bytes(0x3A) for n in (M * ld, rows * nk, rows * nv))
        if fused:
            L.vra_stack_op_gemm_kv(ad.ptr, K + pad, wd.ptr, out.ptr, ld, kc.ptr, vc.ptr, sd.ptr, M, N, K, nq, nk, dt, 0)
        else:
            L.vra_stack_op_gemm(ad.ptr, K + pad, wd.ptr, 0, out.ptr, ld, 0, M, N, K, 1.0, None, 0, None, None, None, 0, 0.0, dt, 0)
            at = lambda c: out.ptr.value + c * es if hasattr(out.ptr, "value") else out.ptr + c * es
            L.vra_stack_op_kv_store(at(nq), at(nq + nk), ld, kc.ptr, vc.ptr, sd.ptr, M, nk, nv, dt, 0)
        check()
        return out.numpy(word, (M, ld))[:, :nq], kc.numpy(word, (rows, nk)), vc.numpy(word, (rows, nv))

    got, want = run(True), run(False)
    assert all(np.array_equal(g, v) for g, v in zip(got, want))
    ref = a[:, :K].astype(np.float64) @ w.astype(np.float64).T
    wide = lambda b: b.view(np.float32) if dt == F32 else (b.astype(np.uint32) << 16).view(np.float32)
    on = slots >= 0
    # float32 sums of K products, and half a unit of the eighth bit where the row is rounded to bf16
    tol = 2e-6 if dt == F32 else 2.0 ** -8
    assert rel(wide(got[0]), ref[:, :nq]) < tol and rel(wide(got[1][slots[on]]), ref[on][:, nq:nq + nk]) < tol and rel(wide(got[2][slots[on]]), ref[on][:, nq + nk:]) < tol
    others = np.setdiff1d(np.arange(rows), slots[on])
    assert (got[1][others].view(np.uint8) == 0x3A).all() and (got[2][others].view(np.uint8) == 0x3A).all()


def test_columns_beyond_the_product_are_refused():
    L = _lib.load()
    x = empty(4096)
    for kv_from, kv_k in ((0, 16), (16, 0), (16, 48), (64, 16)):
        L.vra_stack_op_gemm_kv(x.ptr, 64, x.ptr, x.ptr, 64, x.ptr, x.ptr, x.ptr, 1, 64, 64, kv_from, kv_k, BF16, 0)
        with pytest.raises(RuntimeError, match="cache columns"):
            check()
