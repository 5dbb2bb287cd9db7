"""The 256 x 256, 192 x 256 and 192 x 128 tiles of the row-major prompt GEMM (csrc/gemm_rows.cuh): the bits of the 64 x 128 tile, which the other tests compare with the oracle."""
import ctypes as C

import numpy as np
import pytest

from tests.util import BF16, F16, rand_dt, rng
from vllm_rs_amd import _lib, ops

pytestmark = pytest.mark.gpu


# rows that end in the first or second 64 of either half of a tile and just behind it, columns that leave waves without any, K of one pair of steps and more
@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("M", [33, 65, 129, 200, 256, 257, 530])
@pytest.mark.parametrize("K", [128, 384, 1024])
@pytest.mark.parametrize("form", ["plain", "bias f32", "residual", "segments", "pair"])
def test_wide_tile(form, M, K, dt):
    r = rng(M + K + dt)
    pair, ns = form == "pair", {"segments": [272, 16, 528], "pair": [144] * 2}.get(form, [560])
    x, ws = rand_dt(r, (M, K), dt), [rand_dt(r, (n, K), dt, 0.05) for n in ns]
    bias = [rand_dt(r, (n,), dt, 0.2) if form in ("bias f32", "segments") else None for n in ns]
    res, f32 = rand_dt(r, (M, ns[0]), dt) if form == "residual" else None, form == "bias f32"
    xd, wd, bd = ops.dev(x), [ops.dev(w) for w in ws], [ops.dev(b) if b is not None else None for b in bias]
    rd = ops.dev(res) if res is not None else None

    def run(tile):
        outs = [ops.DevBuf((M + 1) * n * 4).fill_bytes(0) for n in ns]
        ptrs = [(C.c_void_p * len(ns))(*[b.ptr if b else None for b in bufs]) for bufs in (wd, bd, outs)]
        ops.lib().vra_dense_gemm_tile(tile, xd.ptr, ptrs[0], ptrs[1], (C.c_int32 * len(ns))(*ns), len(ns), int(pair), rd.ptr if rd else None, ptrs[2],
                                      int(f32), M, K, dt, 0)
        ops.check_error()
        return [o.numpy(np.float32 if f32 else np.uint16, (M + 1, n)) for o, n in zip(outs, ns)][:1 if pair else None]
    one, wide = run(0x12), run(0x44)
    assert all(g[:M].any() and not g[M].any() for g in wide)  # something in every tensor, nothing beyond the rows
    assert all(np.array_equal(a, b) for a, b in zip(wide, one))


# rows that end in the first or last of a tile's four wave rows of 48 and just behind, one and several tiles, K of one step, fewer than the buffers and more
@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("M", [33, 48, 49, 97, 145, 192, 193, 400])
@pytest.mark.parametrize("K", [64, 192, 1024])
@pytest.mark.parametrize("pair", [False, True])
@pytest.mark.parametrize("tile", [0x32, 0x34])
def test_tile_of_192_rows(tile, pair, M, K, dt):
    if tile == 0x34 and K % 128:
        K += 64
    r = rng(M + K + dt)
    ns = [144] * 2 if pair else [272, 16, 304]
    x, ws = rand_dt(r, (M, K), dt), [rand_dt(r, (n, K), dt, 0.05) for n in ns]
    xd, wd = ops.dev(x), [ops.dev(w) for w in ws]

    def run(tile):
        outs = [ops.DevBuf((M + 1) * n * 2).fill_bytes(0) for n in ns]
        ptrs = [(C.c_void_p * len(ns))(*[b.ptr for b in bufs]) for bufs in (wd, outs)]
        ops.lib().vra_dense_gemm_tile(tile, xd.ptr, ptrs[0], (C.c_void_p * len(ns))(), (C.c_int32 * len(ns))(*ns), len(ns), int(pair), None, ptrs[1], 0, M, K, dt, 0)
        ops.check_error()
        return [o.numpy(np.uint16, (M + 1, n)) for o, n in zip(outs, ns)][:1 if pair else None]
    one, tall = run(0x12), run(tile)
    assert all(g[:M].any() and not g[M].any() for g in tall)
    assert all(np.array_equal(a, b) for a, b in zip(tall, one))


@pytest.mark.parametrize("M,N,K", [(70, 40, 128), (257, 300, 256), (400, 513, 384)])
@pytest.mark.parametrize("scatter", [False, True])
def test_wide_tile_of_a_layer_stack(M, N, K, scatter):
    """f32 outputs off 16 bytes, rows scattered with holes"""
    L = _lib.load()
    r = rng(M + N)
    xd, wd = ops.dev(rand_dt(r, (M, K), BF16)), ops.dev(rand_dt(r, (N, K), BF16, 0.05))
    dst = np.arange(M - 1, -1, -1, dtype=np.int32)
    dst[::3] = -1
    dd = ops.dev(dst.view(np.uint32)) if scatter else None

    def run(tile):
        out = ops.DevBuf((M + 1) * N * 4).fill_bytes(0)
        L.vra_stack_op_gemm_tile(tile, xd.ptr, K, wd.ptr, 0, out.ptr, N, 1, M, N, K, None, None, 0, dd.ptr if dd else None, 0, 0.0, 0)
        ops.check_error()
        return out.numpy(np.float32, (M + 1, N))
    one, wide = run(0x12), run(0x44)
    assert np.array_equal(wide, one) and wide[:M].any() and not wide[M].any()
    assert not scatter or not wide[np.setdiff1d(np.arange(M), dst)].any()


@pytest.mark.parametrize("tile", [0x12, 0x22, 0x24])
@pytest.mark.parametrize("rows128", [1, 3, 17, 33])
@pytest.mark.parametrize("N", [40, 300, 640, 1160])
def test_grouped_rows_reach_every_tile(N, rows128, tile):
    """tile rows around whole rounds of pairs by eight XCDs, empty ones at the end and between, tile columns in one part and in several, the last one short; every product of a row is
    a sum of 64 bf16 products in f32: 2e-6 of the result's norm (a chain of 64 roundings), rows of empty tiles are left alone"""
    L = _lib.load()
    r = rng(N + rows128 + tile)
    K, E, rows = 64, 5, rows128 * 128
    x = (r.standard_normal((rows, K)).astype(np.float32).view(np.uint32) & 0xFFFF0000).view(np.float32)  # bf16 values
    w = (r.standard_normal((E, N, K)).astype(np.float32).view(np.uint32) & 0xFFFF0000).view(np.float32)
    group = r.integers(0, E, rows128).astype(np.int32)
    group[r.random(rows128) < 0.2] = -1
    group[rows128 - rows128 // 4:] = -1
    bits = lambda a: ops.dev((a.view(np.uint32) >> 16).astype(np.uint16))
    gd = ops.dev(np.repeat(group, 128 // ((tile >> 4) * 64)).view(np.uint32))
    xd, wd, out = bits(x), bits(w), ops.DevBuf(rows * N * 4).fill_bytes(0)
    L.vra_stack_op_gemm_tile(tile, xd.ptr, K, wd.ptr, N * K, out.ptr, N, 1, rows, N, K, gd.ptr, None, 0, None, 0, 0.0, 0)
    ops.check_error()
    got = out.numpy(np.float32, (rows, N)).astype(np.float64)
    of_row = np.repeat(group, 128)
    ref = np.zeros((rows, N))
    for e in range(E):
        ref[of_row == e] = x[of_row == e].astype(np.float64) @ w[e].astype(np.float64).T
    assert (got[of_row < 0] == 0).all()
    assert np.linalg.norm(got - ref) <= 2e-6 * max(np.linalg.norm(ref), 1e-30)


# 12, 13, 20 and 24 tile rows: two equal groups, a short last one, the last of two groups, three
@pytest.mark.parametrize("tile,M", [(0x12, 705), (0x12, 769), (0x12, 1217), (0x12, 1473), (0x22, 1537), (0x22, 2945), (0x32, 2305), (0x24, 1537), (0x34, 2305)])
@pytest.mark.parametrize("ns", [[560], [272, 16, 304]])
def test_groups_of_tile_rows_reach_every_tile(ns, tile, M):
    """the tile rows in several groups: the bits of the same rows in pieces of one group"""
    K = 128
    r = rng(M + tile)
    x, ws = rand_dt(r, (M, K), F16), [rand_dt(r, (n, K), F16, 0.05) for n in ns]
    xd, wd = ops.dev(x), [ops.dev(w) for w in ws]

    def run(row, rows, t):
        outs = [ops.DevBuf((rows + 1) * n * 2).fill_bytes(0) for n in ns]
        ptrs = [(C.c_void_p * len(ns))(*[b.ptr for b in bufs]) for bufs in (wd, outs)]
        ops.lib().vra_dense_gemm_tile(t, xd.ptr + row * K * 2, ptrs[0], (C.c_void_p * len(ns))(), (C.c_int32 * len(ns))(*ns), len(ns), 0, None, ptrs[1], 0, rows, K, F16, 0)
        ops.check_error()
        got = [o.numpy(np.uint16, (rows + 1, n)) for o, n in zip(outs, ns)]
        assert not any(g[rows].any() for g in got)
        return [g[:rows] for g in got]
    step = 512
    pieces = [run(row, min(step, M - row), 0x44) for row in range(0, M - 33, step)]  # (the last piece takes what would be too short for one)
    done = sum(len(p[0]) for p in pieces)
    if done < M:
        pieces.append([g[-(M - done):] for g in run(M - 64, 64, 0x44)])
    whole = run(0, M, tile)
    for i, g in enumerate(whole):
        assert np.array_equal(g, np.concatenate([p[i] for p in pieces])) and g.any(axis=1).all()


@pytest.mark.parametrize("tile", [0x32, 0x34, 0x44])
@pytest.mark.parametrize("M,N,K", [(70, 64, 128), (257, 288, 256), (400, 544, 384)])
@pytest.mark.parametrize("form", ["gather", "gated", "gated gather", "bf16"])
def test_tiles_of_a_layer_stack(form, M, N, K, tile):
    """gathered rows with holes, the gated epilogue, 16-bit outputs: the bits of the 64 x 128 tile"""
    L = _lib.load()
    r = rng(M + N + tile)
    rows = M + 31
    xd, wd = ops.dev(rand_dt(r, (rows, K), BF16)), ops.dev(rand_dt(r, (N, K), BF16, 0.05))
    src = r.integers(0, rows, M).astype(np.int32)
    src[::5] = -1
    gather, gated, f32 = "gather" in form, "gated" in form, form == "gather"
    n = N // 2 if gated else N
    sd = ops.dev(src.view(np.uint32)) if gather else None

    def run(t):
        out = ops.DevBuf((M + 1) * n * 4).fill_bytes(0)
        L.vra_stack_op_gemm_tile(t, xd.ptr, K, wd.ptr, 0, out.ptr, n, int(f32), M, N, K, None, sd.ptr if sd else None, rows if sd else 0, None, int(gated), 7.0, 0)
        ops.check_error()
        return out.numpy(np.float32 if f32 else np.uint16, (M + 1, n))
    one, other = run(0x12), run(tile)
    assert np.array_equal(other, one) and other[:M].any() and not other[M].any()
    assert not gather or not other[:M][src < 0].any()


@pytest.mark.parametrize("tile,K,grouped", [(0x34, 192, False), (0x44, 192, False), (0x34, 64, False), (0x32, 128, True), (0x34, 128, True), (0x44, 128, True), (0x14, 128, False)])
def test_tiles_that_do_not_fit_are_refused(tile, K, grouped):
    """K steps of two phases come in pairs; only tiles of 64 and 128 rows look at their row groups"""
    L = _lib.load()
    M, N = 768, 128
    xd, wd, out = ops.dev(np.zeros((M, K), np.uint16)), ops.dev(np.zeros((N, K), np.uint16)), ops.DevBuf(M * N * 4).fill_bytes(0x55)
    gd = ops.dev(np.zeros(M // 64, np.uint32)) if grouped else None
    L.vra_stack_op_gemm_tile(tile, xd.ptr, K, wd.ptr, 0, out.ptr, N, 1, M, N, K, gd.ptr if gd else None, None, 0, None, 0, 0.0, 0)
    assert L.vra_last_error().decode()
    L.vra_clear_error()
    if not grouped:
        L.vra_dense_gemm_tile(tile, xd.ptr, (C.c_void_p * 1)(wd.ptr), (C.c_void_p * 1)(), (C.c_int32 * 1)(N), 1, 0, None, (C.c_void_p * 1)(out.ptr), 0, M, K, BF16, 0)
        assert L.vra_last_error().decode()
        L.vra_clear_error()
    L.vra_device_sync()
    assert (out.numpy(np.uint8, (M * N * 4,)) == 0x55).all()
