"""Down projections of 64..96 and 129..160 rows in a model's step: kernel M where it is quicker than kernel W's row blocks."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.test_gpu_kernels import wna16_on
from tests.util import BF16, F16, assert_close_dt, make_quant, rand_dt, rng
from vllm_rs_amd import ops

pytestmark = pytest.mark.gpu


def test_where_the_line_lies():
    pick = lambda m, k, n, awq=0, gs=128: chr(ops.lib().vra_wna16_down_kernel(m, k, n, gs, awq, 0, 1))
    entry = lambda m, k, n, awq=0, gs=128: chr(ops.lib().vra_wna16_kernel(0, m, k, n, gs, awq, 0, 0, 1))
    for m in (64, 96, 129, 150, 160):  # quicker on M, kept on W by the entry point
        assert pick(m, 14336, 4096) == "M" and entry(m, 14336, 4096) == "W"
    assert pick(150, 18944, 3584, 1) == "M" and pick(150, 8192, 8192) == "M"
    for m, k, n, awq in ((150, 14336, 1024, 0), (150, 8192, 3584, 0), (64, 18944, 3584, 1), (63, 14336, 4096, 0), (33, 14336, 4096, 0), (32, 14336, 4096, 0)):
        assert pick(m, k, n, awq) == "W"
    for m, k, n, gs in ((100, 14336, 4096, 128), (161, 14336, 4096, 128), (300, 14336, 4096, 128), (150, 4096, 4096, 128), (8, 14336, 4096, 128), (1, 14336, 4096, 128),
                        (150, 14336, 4096, 64)):  # everything else: as the entry point
        assert pick(m, k, n, 0, gs) == entry(m, k, n, 0, gs)


# the rows at the edges of the range and of kernel M's blocks of 32 and 160, the last columns of a tile missing
@pytest.mark.parametrize("M", [64, 65, 96, 129, 150, 160])
@pytest.mark.parametrize("dt,awq,K,N", [(BF16, False, 8192, 8192), (F16, True, 18944, 4112), (F16, False, 14336, 4080)])
def test_kernel_m_bias_residual(dt, awq, K, N, M):
    r = rng(M + N + awq)
    q, x, bias, res = make_quant(r, K, N, 128, dt, awq), rand_dt(r, (M, K), dt), rand_dt(r, (N,), dt), rand_dt(r, (M, N), dt)
    z = q["zeros"] if awq else None
    ref, g0 = orc.wna16_gemm(x, q["idx"], z, q["scales"], 128, dt, bias, res), orc.from_dt(orc.wna16_gemm(x, q["idx"], z, q["scales"], 128, dt), dt)
    mag = np.maximum(np.abs(g0), np.abs(g0 + orc.from_dt(bias, dt)[None, :]))
    # (three roundings, each to the neighbouring value at most: the bound of the other tests of this kernel)
    assert_close_dt(wna16_on("M", x, q, M, K, N, 128, dt, awq, bias, res), ref, dt, max_ulp=3.0, name=f"down on M {M} x {N}", mag=mag)


# as the model's step runs it, the residual in the output's own rows: the bits of two buffers, where K is in one slice and in several that meet in the last one's
# epilogue (256 CUs: 160 tiles of 128 columns leave no room for a second slice, 9 and 32 do)
@pytest.mark.parametrize("M", [64, 96, 129, 160])
@pytest.mark.parametrize("dt,awq,K,N", [(BF16, False, 4224, 20480), (F16, True, 18944, 1040), (BF16, False, 14336, 4096)])
def test_kernel_m_in_place(dt, awq, K, N, M):
    r = rng(M + N + K)
    q, x, res = make_quant(r, K, N, 128, dt, awq), rand_dt(r, (M, K), dt), rand_dt(r, (M, N), dt)
    w = ops.marlin_weight_repack(ops.dev(q["qweight"]), q["qweight"].shape, 4, awq)
    xd, sc, z, out = ops.dev(x), ops.dev(q["scales"]), ops.dev(q["qzeros"]) if awq else None, ops.dev(np.concatenate([res, res[:1]]))  # (a row behind it)
    ops.lib().vra_wna16_gemm_on(ord("M"), xd.ptr, w.ptr, sc.ptr, z.ptr if awq else None, None, None, None, None, out.ptr, out.ptr, M, K, N, 128, int(awq), dt, 0)
    ops.check_error()
    got = out.numpy(np.uint16, (M + 1, N))
    assert np.array_equal(got[:M], wna16_on("M", x, q, M, K, N, 128, dt, awq, None, res)) and np.array_equal(got[M], res[0])
