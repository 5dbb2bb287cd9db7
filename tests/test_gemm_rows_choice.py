"""The tile that the row-major prompt GEMM takes (csrc/gemm_rows.cuh) against the measured times of all tiles, weights from memory."""
import ctypes as C
import os

import numpy as np

from vllm_rs_amd import _lib

TIMES = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "profiles", "gemm_rows_tile_times.txt")
TILES = (0x12, 0x22, 0x32, 0x24, 0x34, 0x44)


def test_chosen_tile_is_near_the_fastest_and_no_slower_than_before():
    L = _lib.load()
    rows = [line.split() for line in open(TIMES) if line[0].isdigit()]
    assert len(rows) > 700
    behind = []
    for v in rows:
        m, n, k = (int(x) for x in v[:3])
        times = {t: float(x) for t, x in zip(TILES, v[4:]) if x != "-"}
        tile = L.vra_dense_gemm_tile_choice(m, (C.c_int32 * 1)(n), 1, k)
        # (one sweep's medians of three: two of them differ by up to 4 %)
        assert times[tile] <= 1.04 * float(v[3]), (m, n, k, hex(tile), v)
        assert times[tile] <= 1.10 * min(times.values()), (m, n, k, hex(tile), times)
        behind.append(times[tile] / min(times.values()))
    assert np.mean(behind) < 1.002


def test_tiles_of_two_phases_need_whole_pairs_of_k_steps():
    L = _lib.load()
    for k in (64, 192, 2112):
        for m in (2048, 4096, 8192):
            assert L.vra_dense_gemm_tile_choice(m, (C.c_int32 * 2)(8192, 8192), 2, k) in (0x12, 0x22, 0x32, 0x24)
    assert L.vra_dense_gemm_tile_choice(8192, (C.c_int32 * 1)(8192), 1, 2048) == 0x44
    assert L.vra_dense_gemm_tile_choice(0, (C.c_int32 * 1)(8192), 1, 2048) == 0
