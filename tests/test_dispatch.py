"""Which kernel a shape runs on, where that is decided without a GPU (vra_wna16_kernel)."""
import ctypes
import os
import subprocess
import sys

import pytest

from vllm_rs_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
QUERY = "from vllm_rs_amd import ops; print(''.join(ops.wna16_kernel(%d, m, 4096, 14336, 128, has_norm=True) for m in (16, 32, 33, 64)))"


def kernels(pair, **env):
    """the letters for 16, 32, 33 and 64 rows in a process of its own: the tuning aids are read once"""
    out = subprocess.run([sys.executable, "-c", QUERY % pair], cwd=ROOT, env=dict(os.environ, **env), capture_output=True, text=True, check=True)
    return out.stdout.strip()


@pytest.mark.parametrize("pair", [0, 1])
def test_rows_limit_of_kernel_w_holds_for_single_products_and_pairs(pair):
    assert kernels(pair) == "WWWW"
    short = kernels(pair, VRA_GEMV_W_MAX_ROWS="32")
    assert short[:2] == "WW" and "W" not in short[2:], short


def test_linear_recurrence_stays_within_the_default_lds():
    """its launch raises no limit, so 64 KB is all it may ask for, at every key size and form"""
    lds = _lib.load().vra_stack_op_linear_scan_lds
    assert max(lds(dim, dim, 16, B, n) for dim in range(1, 257) for B in (1, 64) for n in (0, 1, 5, 100)) <= 64 * 1024
    assert lds(0, 1, 1, 1, 0) < 0 and lds(257, 1, 1, 1, 0) < 0


def test_rotary_and_cache_store_stay_within_the_default_lds():
    """as above: what is staged for a group of 8 tokens and what the kernel keeps beside it; prompts of many tokens and heads are still taken in groups"""
    plan, lds = _lib.load().vra_rope_cache_prefill_slices, ctypes.c_int32()
    for kv_heads in (1, 3, 8, 12, 16, 24, 31, 32, 33, 40, 64, 128):
        for dim in (64, 80, 128, 256):
            for tokens in (100, 256, 700, 1024, 2100, 4096, 8184, 8185, 8192, 30000):
                for kv_dtype in (0, 3):
                    slices = plan(tokens, kv_heads, dim, 64, kv_dtype, ctypes.addressof(lds))
                    assert 0 <= slices <= kv_heads and lds.value <= 64 * 1024, (kv_heads, dim, tokens, kv_dtype, slices, lds.value)
                    assert (slices > 0) == (tokens >= 1024 or tokens >= 256 and tokens * kv_heads * dim >= 384 << 10)
                    assert plan(tokens, kv_heads, dim, 20, kv_dtype, None) == 0  # (pages off 8 tokens)
    assert [plan(n, 8, 128, 64, 0, None) for n in (1200, 1500, 3000, 8192)] == [7, 6, 3, 1]


def test_no_more_logit_rows_in_place_than_the_callers_array_holds():
    """a step padded to its bucket computes more rows than the caller asked for: those go to the device's rows only"""
    rows = _lib.load().vra_logit_rows_in_place
    for seqs in range(1, 41):
        for step in range(seqs, 65):
            assert rows(0, seqs, step) == (seqs if step == seqs else 0)
            assert rows(7, seqs, step) == 7  # (wanted rows: as many as the step's head computes)


@pytest.mark.parametrize("dim", [4, 32, 64, 128, 256])
def test_linear_recurrence_stages_one_token_for_one(dim):
    """a decode step's workgroups stage one token: q, k, decays, value and output of it and three numbers"""
    P = max(1, dim // 4)
    assert _lib.load().vra_stack_op_linear_scan_lds(dim, dim, 16, 8, 1) == 4 * (3 * dim + 2 * (256 // P) + 3)


@pytest.mark.parametrize("experts", [4, 16, 64])
@pytest.mark.parametrize("pairs", [1, 40, 1000, 16384])
def test_expert_rows(pairs, experts):
    """the row space a mixture sizes its buffers by: what its granule can need and no more, and enough for every shorter step"""
    rows = _lib.load().vra_stack_op_expert_rows
    for tiles in (0, 1):
        pad = 16 if pairs // experts < (96 if tiles else 128) else (128 if tiles else 64)
        assert pairs + experts * (pad - 1) <= rows(pairs, experts, tiles) < pairs + experts * (pad - 1) + pad
        assert rows(pairs, experts, tiles) >= max(rows(n, experts, tiles) for n in range(1, pairs + 1, max(1, pairs // 97)))


# us, 32 columns a workgroup / 16 (MI355X, weights not in any cache)
@pytest.mark.parametrize("M,N,K,want", [
    (8, 2048, 8192, 16),  # 22.9 / 14.6
    (32, 2048, 256, 16),  # 5.3 / 4.4
    (17, 3072, 8192, 32),  # 25.4 / 31.1
    (32, 4000, 4096, 32),  # 15.9 / 18.1
    (32, 3072, 512, 32),  # 5.6 / 6.2
    (16, 6144, 4096, 32),  # 16.7 / 19.2
    (16, 4096, 4096, 16),  # 16.1 / 11.9
    (8, 6144, 512, 32),  # 5.1 / 5.6
])
def test_columns_of_few_row_products(M, N, K, want):
    L = _lib.load()
    assert L.vra_stack_op_gemm_few_columns(M, N, 1, 0) == want and L.vra_stack_op_gemm_few_columns(M, N, 1, 1) == 32
