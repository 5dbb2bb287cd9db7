"""The 192 x 256 tile of the dense prompt GEMM (csrc/gemm_dense.cuh): the bits of the 256 x 256 tile, which the other tests compare with the oracle."""
import ctypes as C

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


# 12, 13 and 21 tile rows of 192 (two groups, a short second one, three); 12 and 20 of 256
@pytest.mark.parametrize("tile,M", [(192, 2113), (192, 2305), (192, 3841), (256, 2817), (256, 4865), (128, 2817)])
def test_groups_of_tile_rows_reach_every_tile(tile, M):
    """the tile rows in several groups: the bits of the same rows in pieces of one group"""
    K, NV, step = 128, 528, 1024
    r = rng(M + tile)
    x, wd = ops.dev(rand_dt(r, (M, K), F16)), ops.dev(rand_dt(r, (NV, K), F16, 0.05))

    def run(row, rows, t):
        out = ops.DevBuf((rows + 1) * NV * 2).fill_bytes(0)
        ops.lib().vra_dense_frag_gemm(x.ptr + row * K * 2, wd.ptr, None, None, out.ptr, rows, K, NV, 0, F16, t, 0)
        ops.check_error()
        got = out.numpy(np.uint16, (rows + 1, NV))
        assert not got[rows].any()
        return got[:rows]
    whole = run(0, M, tile)
    assert np.array_equal(whole, np.concatenate([run(row, min(step, M - row), 256) for row in range(0, M, step)])) and whole.any(axis=1).all()


@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("M", [50, 193, 700])
@pytest.mark.parametrize("ns", [[64, 64, 64], [320, 64, 144], [512, 128, 128], [256, 272]])
@pytest.mark.parametrize("tile", [128, 192, 256, 256 | 2 << 16])
def test_segments(tile, ns, M, dt):
    """q, k and v side by side, each with a bias and an output of its own: the bits of one tensor of all columns"""
    K = 256
    r = rng(M + sum(ns) + dt)
    NV = sum(ns)
    x, wd = ops.dev(rand_dt(r, (M, K), dt)), ops.dev(rand_dt(r, (NV, K), dt, 0.05))
    bias = rand_dt(r, (NV,), dt)
    one = ops.DevBuf(M * NV * 2).fill_bytes(0)
    bd = ops.dev(bias)
    ops.lib().vra_dense_frag_gemm(x.ptr, wd.ptr, bd.ptr, None, one.ptr, M, K, NV, 0, dt, tile, 0)
    ops.check_error()
    cut = np.cumsum([0] + ns)
    bds = [ops.dev(bias[a:b].copy()) for a, b in zip(cut, cut[1:])]
    outs = [ops.DevBuf((M + 1) * n * 2).fill_bytes(0) for n in ns]
    ops.lib().vra_dense_frag_gemm_segments(x.ptr, wd.ptr, (C.c_void_p * len(ns))(*[b.ptr for b in bds]), (C.c_int32 * len(ns))(*ns), len(ns),
                                           (C.c_void_p * len(ns))(*[o.ptr for o in outs]), M, K, dt, tile, 0)
    ops.check_error()
    want = one.numpy(np.uint16, (M, NV))
    for o, a, b in zip(outs, cut, cut[1:]):
        got = o.numpy(np.uint16, (M + 1, b - a))
        assert np.array_equal(got[:M], want[:, a:b]) and got[:M].any() and not got[M].any()


def test_segments_that_do_not_fit_are_refused():
    L = ops.lib()
    x, wd, out = ops.DevBuf(256 * 128 * 2).zero(), ops.DevBuf(256 * 128 * 2).zero(), ops.DevBuf(256 * 256 * 2)
    for ns in ([48, 64], [64, 40], [64, 64, 64, 64], []):  # (a segment begins at a multiple of 64 columns, ends at one of 16; at most three)
        L.vra_dense_frag_gemm_segments(x.ptr, wd.ptr, (C.c_void_p * 4)(), (C.c_int32 * 4)(*ns), len(ns), (C.c_void_p * 4)(*[out.ptr] * 4), 64, 128, BF16, 192, 0)
        assert L.vra_last_error().decode()
        L.vra_clear_error()
