"""The row-major prompt GEMM on two tiles (csrc/gemm_rows.cuh gemm_rows_mixed_kernel), as the decoders and as the layer stacks launch it: the bits of the
64 x 128 tile, which the other tests compare with the oracle."""
import ctypes as C

import numpy as np
import pytest

from oracle import oracle as orc
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
    one = product(0x12, x, w, [None], None, M, K, dt, False, False)
    assert np.array_equal(product(tile, x, w, [None], None, M, K, dt, False, False), one)
    xd, wd, out = ops.dev(x), ops.dev(w[0]), ops.DevBuf((M + 1) * N * 2).fill_bytes(0)  # (the entry point, which chooses itself)
    ops.lib().vra_dense_gemm(xd.ptr, wd.ptr, None, out.ptr, M, K, N, dt, dt, 0)
    ops.check_error()
    assert np.array_equal(out.numpy(np.uint16, (M + 1, N)), one)


# --- a layer stack's products: sums in f32 and bf16, rows scattered with holes, gated pairs (half as many columns), key and value columns to their cache rows
FORMS = ("f32", "bf16", "off 16 bytes", "scatter", "gated", "kv")
NO_SLOT = 0x3A


def stack_product(tile, form, ad, wd, dd, sd, M, N, K, nq, nk, rows):
    """every output's bytes; tile 0: the choice by size"""
    L, f32 = _lib.load(), form in ("f32", "scatter")
    ldo, es = (N // 2 if form == "gated" else N), 4 if f32 else 2
    out = ops.DevBuf((M + 1) * ldo * es).fill_bytes(NO_SLOT)
    if form == "kv":
        kc, vc = ops.DevBuf(rows * nk * 2).fill_bytes(NO_SLOT), ops.DevBuf(rows * (N - nq - nk) * 2).fill_bytes(NO_SLOT)
        L.vra_stack_op_gemm_kv_tile(tile, ad.ptr, K, wd.ptr, out.ptr, ldo, kc.ptr, vc.ptr, sd.ptr, M, N, K, nq, nk, BF16, 0)
        ops.check_error()
        return [out.numpy(np.uint16, (M + 1, ldo))[:, :nq], kc.numpy(np.uint16, (rows, nk)), vc.numpy(np.uint16, (rows, N - nq - nk))]
    tail = (dd.ptr if form == "scatter" else None, int(form == "gated"), 1.5)
    if tile:
        L.vra_stack_op_gemm_tile(tile, ad.ptr, K, wd.ptr, 0, out.ptr, ldo, int(f32), M, N, K, None, None, 0, *tail, 0)
    else:
        L.vra_stack_op_gemm(ad.ptr, K, wd.ptr, 0, out.ptr, ldo, int(f32), M, N, K, 1.0, None, 0, None, None, *tail, BF16, 0)
    ops.check_error()
    return [out.numpy(np.float32 if f32 else np.uint16, (M + 1, ldo))]


def stack_operands(r, M, N, K):
    rows = M + 40
    dst, slots = np.arange(M - 1, -1, -1, dtype=np.int32), r.permutation(rows)[:M].astype(np.int64)
    dst[::3], slots[1::5] = -1, -1
    return [ops.dev(rand_dt(r, (M, K), BF16)), ops.dev(rand_dt(r, (N, K), BF16, 0.05)), ops.dev(dst.view(np.uint32)), ops.dev(slots.view(np.uint32))], dst, slots, rows


def check_untouched(got, form, M, dst, slots):
    untouched = lambda a: not a.size or (np.ascontiguousarray(a).view(np.uint8) == NO_SLOT).all()
    assert untouched(got[0][M])
    assert form != "scatter" or untouched(got[0][:M][np.setdiff1d(np.arange(M), dst)])
    for cache in got[1:]:
        assert untouched(cache[np.setdiff1d(np.arange(len(cache)), slots)]) and not untouched(cache[slots[slots >= 0]])


# rows as above; key columns begin and value columns begin inside a tile, on the large tile, on the small one and in the strip behind it
@pytest.mark.parametrize("M", [256, 257, 511, 530])
@pytest.mark.parametrize("form", FORMS)
def test_two_tiles_of_a_layer_stack(form, M):
    K, N = 256, {"gated": 800, "off 16 bytes": 781}.get(form, 784)
    args, dst, slots, rows = stack_operands(rng(M + N), M, N, K)
    for nq, nk in ((264, 248), (520, 8), (40, 8)) if form == "kv" else ((0, 0),):
        one = stack_product(0x12, form, *args, M, N, K, nq, nk, rows)
        assert one[0][:M].any()
        for columns in (1, 3, 4):
            got = stack_product(0x44 | columns << 8, form, *args, M, N, K, nq, nk, rows)
            assert all(np.array_equal(a, b) for a, b in zip(got, one)), (nq, columns)
            check_untouched(got, form, M, dst, slots)


# by size: 8 of 12 tile columns are large
@pytest.mark.parametrize("form", [f for f in FORMS if f != "off 16 bytes"])
def test_two_tiles_of_a_layer_stack_by_size(form):
    M, N, K = 8192, 3072, 2048
    tile = ops.lib().vra_dense_gemm_tiles_choice(M, N, K)
    assert tile & 0xff == 0x44 and 0 < tile >> 8 < N // 256
    args, dst, slots, rows = stack_operands(rng(M), M, N, K)
    one, got = (stack_product(t, form, *args, M, N, K, 2048, 512, rows) for t in (0x12, 0))
    assert all(np.array_equal(a, b) for a, b in zip(got, one))
    check_untouched(got, form, M, dst, slots)


# a bias, loaded once for all rows of a wave: the sums without it and the bias in f32, bit for bit (columns off 16 bytes; whole pieces on one tile and on two)
@pytest.mark.parametrize("M,N,K", [(40, 70, 64), (530, 781, 256), (530, 784, 256), (2120, 3076, 1024), (8192, 3072, 128)])
def test_bias_of_a_layer_stack(M, N, K):
    r = rng(M + N)
    a, w, bias = ops.dev(rand_dt(r, (M, K), BF16)), ops.dev(rand_dt(r, (N, K), BF16, 0.05)), r.standard_normal(N).astype(np.float32)
    bd = ops.dev(bias)

    def run(b, f32):
        out = ops.DevBuf((M + 1) * N * 4).fill_bytes(NO_SLOT)
        ops.lib().vra_stack_op_gemm_ex(a.ptr, K, w.ptr, out.ptr, N, f32, M, N, K, 1.0, b, 0, 0, 1, 0, 0, 0, BF16, 0)
        ops.check_error()
        got = out.numpy(np.float32 if f32 else np.uint16, (M + 1, N))
        assert (got[M].view(np.uint8) == NO_SLOT).all()
        return got[:M]

    want = run(None, 1) + bias
    assert np.array_equal(run(bd.ptr, 1), want) and np.array_equal(run(bd.ptr, 0), orc.to_dt(want, BF16))


def test_two_tiles_of_a_layer_stack_are_refused():
    """rows in groups, few rows, half a pair of K steps, more columns than there are, another tile, a function that is not built for it"""
    L = _lib.load()
    x = ops.DevBuf(1024 * 1024).fill_bytes(0)
    gd = ops.dev(np.zeros(16, np.uint32))
    for tile, M, K, group in ((0x144, 512, 128, gd.ptr), (0x144, 255, 128, None), (0x144, 512, 192, None), (0x344, 512, 128, None), (0x124, 512, 128, None)):
        L.vra_stack_op_gemm_tile(tile, x.ptr, K, x.ptr, 0, x.ptr, 512, 1, M, 512, K, group, None, 0, None, 0, 0.0, 0)
        with pytest.raises(RuntimeError):
            ops.check_error()


def test_refused():
    x, w = np.zeros((512, 192), np.uint16), [np.zeros((512, 192), np.uint16)]
    for M, K, tile in ((255, 128, 0x144), (512, 192, 0x144), (512, 128, 0x344), (512, 128, 0x124)):  # few rows, half a pair of K steps, more columns than there are, another tile
        with pytest.raises(Exception):
            product(tile, x[:M, :K].copy(), [w[0][:, :K].copy()], [None], None, M, K, BF16, False, False)
    assert ops.lib().vra_dense_gemm_tiles_choice(8192, 8192, 2112) & ~0xff == 0 and ops.lib().vra_dense_gemm_tiles_choice(128, 8192, 2048) >> 8 == 0
