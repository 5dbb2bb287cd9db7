"""The 192 x 256 tile of the dense prompt GEMM (csrc/gemm_dense.cuh): the bits of the 256 x 256 tile, which the other tests compare with the oracle."""
import numpy as np
import pytest

from tests.util import BF16, F16, rand_dt, rng
from vllm_rs_amd import ops

pytestmark = pytest.mark.gpu


# rows that end in the first or last of a tile's fragments of 16, in either half of 96 and just behind; columns that leave a wave or half a wave without
# any, K of one pair of steps and more
@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("M", [1, 16, 49, 97, 191, 192, 193, 400])
@pytest.mark.parametrize("K", [128, 384, 1024])
@pytest.mark.parametrize("form,NV", [("plain", 256), ("plain", 528), ("bias residual", 80), ("gate up", 544)])
def test_tile_of_192_rows(form, NV, M, K, dt):
    r = rng(M + K + NV + dt)
    dual, both = form == "gate up", form == "bias residual"
    n = NV // 2 if dual else NV
    x, wd = ops.dev(rand_dt(r, (M, K), dt)), ops.dev(rand_dt(r, (NV, K), dt, 0.05))
    bias, res = (ops.dev(rand_dt(r, (n,), dt)), ops.dev(rand_dt(r, (M, n), dt))) if both else (None, None)

    def run(tile):
        out = ops.DevBuf((M + 1) * n * 2).fill_bytes(0)
        ops.lib().vra_dense_frag_gemm(x.ptr, wd.ptr, bias.ptr if bias else None, res.ptr if res else None, out.ptr, M, K, NV, int(dual), dt, tile, 0)
        ops.check_error()
        return out.numpy(np.uint16, (M + 1, n))
    got, want = run(192), run(256)
    assert np.array_equal(got, want) and got[:M].any() and not got[M].any()
