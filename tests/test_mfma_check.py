"""tools/check_mfma_overlap.py, which the build runs over the kernels' assembly: hazards across branches, loop ends and barriers are seen."""
import os
import sys

import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "tools"))
import check_mfma_overlap as chk  # noqa: E402

MFMA = "\tv_mfma_f32_16x16x32_bf16 v[0:3], v[4:7], v[8:11], v[0:3]\n"
DRAIN = "\ts_nop 7\n\ts_nop 4\n"


@pytest.mark.parametrize("body,violations", [
    ("\tv_mov_b32 v4, v20\n" + MFMA, 1),
    ("\tv_mov_b32 v4, v20\n\ts_nop 1\n" + MFMA, 0),
    ("\tv_mov_b32 v20, v4\n" + MFMA, 0),
    ("\tv_mov_b32 v4, v20\n\ts_barrier\n" + MFMA, 1),
    ("\tv_mov_b32 v4, v20\n\ts_nop 0\n\ts_barrier\n" + MFMA, 0),
    ("\tv_mov_b32 v4, v20\n\ts_cbranch_scc1 .LBB0_1\n" + MFMA + DRAIN + ".LBB0_1:\n", 1),  # the way past a branch
    ("\tv_mov_b32 v4, v20\n\ts_cbranch_scc1 .LBB0_1\n\ts_nop 1\n.LBB0_1:\n" + MFMA, 1),  # the way along it
    ("\tv_mov_b32 v4, v20\n\ts_branch .LBB0_2\n.LBB0_1:\n" + MFMA + DRAIN + ".LBB0_2:\n", 0),
    ("\ts_nop 1\n.LBB0_1:\n" + MFMA + DRAIN + "\tv_permlane32_swap_b32 v20, v11\n\ts_cbranch_scc1 .LBB0_1\n", 1),  # the end of a loop and its head
    (MFMA + "\ts_cbranch_scc1 .LBB0_1\n" + DRAIN + ".LBB0_1:\n\tv_add_f32 v20, v20, v3\n", 1),
    (MFMA + "\ts_cbranch_scc1 .LBB0_1\n" + DRAIN + "\tv_add_f32 v20, v20, v3\n.LBB0_1:\n", 0),
    (MFMA + "\ts_branch .LBB0_1\n\tv_add_f32 v20, v20, v3\n.LBB0_1:\n" + DRAIN + "\tv_add_f32 v20, v20, v3\n", 0),
    (".LBB0_1:\n\tglobal_store_dword v20, v3, s[4:5]\n\ts_nop 1\n" + MFMA + "\ts_cbranch_scc1 .LBB0_1\n" + DRAIN, 1),
    (".LBB0_1:\n" + MFMA + "\ts_cbranch_scc1 .LBB0_1\n" + DRAIN + "\tglobal_store_dword v20, v3, s[4:5]\n", 0),  # the next turn accumulates
    ("\ts_cbranch_scc1 .LBB0_1\n\ts_endpgm\n.LBB0_1:\n\tv_mov_b32 v4, v20\n" + MFMA, 1),  # behind a first way out
    ("\tv_mfma_f32_16x16x32_bf16 v[0:3], v[2:5], v[8:11], v[0:3]\n", 1),
])
def test_hazards(tmp_path, body, violations):
    f = tmp_path / "k.s"
    f.write_text("_Z1kv:\n" + body + "\ts_endpgm\n.Lfunc_end0:\n")
    total, bad = chk.check(str(f))
    assert (total, bad) == (1, violations)
