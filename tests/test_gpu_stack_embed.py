"""Embeddings with sine positions of long prompts (two angles a thread at a time): the bits of the rows one by one."""
import numpy as np
import pytest

from tests.test_gpu_stack import F32, raw, to_dev
from tests.util import BF16, rng
from vllm_rs_amd import ops

pytestmark = pytest.mark.gpu


# rows that end inside a thread's four angles, just behind a workgroup's first and second thousand, and rows not in fours (one angle at a time)
@pytest.mark.parametrize("dt", [BF16, F32])
@pytest.mark.parametrize("W", [4, 516, 1020, 2048, 2052, 4100, 1030])
@pytest.mark.parametrize("positions", [True, False])
def test_long_prompt_equals_rows_one_by_one(W, positions, dt, T=257):
    V = 19
    r = rng(W + dt)
    ids, pos, emb = r.integers(0, V + 2, T).astype(np.uint32), r.integers(0, 9000, T).astype(np.int64), r.standard_normal((V, W)).astype(np.float32)
    inv = raw((10000.0 ** (-np.arange((W + 1) // 2) * 2.0 / W)).astype(np.float32), np.float32) if positions else None
    ed = to_dev(emb, dt)

    def run(ids, pos):
        x = ops.DevBuf((len(ids) + 1) * W * 4).fill_bytes(0)
        ops.lib().vra_stack_op_embed_sinpos(raw(ids, np.uint32).ptr, raw(pos, np.int64).ptr, ed.ptr, inv.ptr if positions else None, x.ptr, len(ids), W, V, dt, 0)
        ops.check_error()
        return x.numpy(np.float32, (len(ids) + 1, W))
    got = run(ids, pos)
    assert not got[T].any()
    for t in (0, 1, 100, T - 1):
        assert np.array_equal(got[t], run(ids[t:t + 1], pos[t:t + 1])[0])


# narrow rows: one angle at a time up to 1023 rows, and beyond where two by two would leave part of a wave idle
@pytest.mark.parametrize("T,W", [(1023, 512), (1024, 512), (1024, 256), (1024, 384), (300, 512)])
def test_narrow_rows_of_long_prompts(T, W):
    test_long_prompt_equals_rows_one_by_one(W, True, BF16, T)
