"""The row-major prompt GEMM on two tiles (csrc/gemm_rows.cuh gemm_rows_mixed_kernel): the bits of the 64 x 128 tile, which the other tests compare with the oracle."""
import ctypes as C

import numpy as np
import pytest

from tests.util import BF16, F16, rand_dt, rng
from vllm_rs_amd import _lib, ops

pytestmark = pytest.mark.gpu


def product(tile, x, ws, bias, res, M, K, dt, pair, f32):
    n = ws[0].shape[0]
    xd, wd, bd, rd = ops.dev(x), [ops.dev(w) for w in ws], [ops.dev(b) if b is not None else None for b in bias], ops.dev(res) if res is not None else None
    outs = [ops.DevBuf((M + 1) * n * 4).fill_bytes(0) for _ in ws]
    ptrs = [(C.c_void_p * len(ws))(*[b.ptr if b else None for b in bufs]) for bufs in (wd, bd, outs)]
    ops.lib().vra_dense_gemm_tile(tile, xd.ptr, ptrs[0], ptrs[1], (C.c_int32 * len(ws))(*[n] * len(ws)), len(ws), int(pair), rd.ptr if rd else None, ptrs[2], int(f32), M, K,
                                  dt, 0)
    ops.check_error()
    return outs[0].numpy(np.float32 if f32 else np.uint16, (M + 1, n))


# rows that end with the last whole 256, within the small tile below it and in the second of two, columns that end inside a tile; the first, some and all columns on
# the large tile (then a strip below or nothing is left)
@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("form", ["plain", "bias f32", "residual", "pair"])
@pytest.mark.parametrize("M", [256, 257, 384, 511, 530, 1100])
@pytest.mark.parametrize("K", [128, 640])
def test_two_tiles(form, M, K, dt):
    r = rng(M + K + dt)
    pair, f32 = form == "pair", form == "bias f32"
    n = 400 if pair else 784  # 800 virtual columns: four tile columns, the last ragged
    x, ws = rand_dt(r, (M, K), dt), [rand_dt(r, (n, K), dt, 0.05) for _ in range(2 if pair else 1)]
    bias = [rand_dt(r, (n,), dt, 0.2) if f32 else None for _ in ws]
    res = rand_dt(r, (M, n), dt) if form == "residual" else None
    one = product(0x12, x, ws, bias, res, M, K, dt, pair, f32)
    assert one[:M].any() and not one[M].any()
    for columns in (1, 3, 4):
        assert np.array_equal(product(0x44 | columns << 8, x, ws, bias, res, M, K, dt, pair, f32), one)


# products that take it by themselves: some tile columns large, more than one round of either tile
@pytest.mark.parametrize("M,N", [(2120, 11264), (1300, 28672)])
def test_chosen_by_size(M, N):
    K, dt = 2048, BF16
    tile = ops.lib().vra_dense_gemm_tiles_choice(M, N, K)
    assert tile & 0xff == 0x44 and 0 < tile >> 8 <= N // 256
    r = rng(M)
    x, w = rand_dt(r, (M, K), dt), [rand_dt(r, (N, K), dt, 0.05)]
    assert np.array_equal(product(tile, x, w, [None], None, M, K, dt, False, False), product(0x12, x, w, [None], None, M, K, dt, False, False))


def test_refused():
    x, w = np.zeros((512, 192), np.uint16), [np.zeros((512, 192), np.uint16)]
    for M, K, tile in ((255, 128, 0x144), (512, 192, 0x144), (512, 128, 0x344), (512, 128, 0x124)):  # few rows, half a pair of K steps, more columns than there are, another tile
        with pytest.raises(Exception):
            product(tile, x[:M, :K].copy(), [w[0][:, :K].copy()], [None], None, M, K, BF16, False, False)
    assert ops.lib().vra_dense_gemm_tiles_choice(8192, 8192, 2112) & ~0xff == 0 and ops.lib().vra_dense_gemm_tiles_choice(128, 8192, 2048) >> 8 == 0
