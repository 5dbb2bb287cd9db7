"""Logits that the head's launch stores in pinned host memory itself (host/engine.cpp pinned_device_view; csrc/gemv.cuh, gemv_dw.cuh, stack_ops.hip `mirror`)
against the copy that an ordinary or an unaligned buffer takes, and the model's own device rows: bit for bit, nothing before or behind them, at the edges of the
heads' forms (1..3 rows, one and two tiles of rows, more rows than they take; 8, 16 and 32 rows of a layer stack, float32).  Which of the two ways a step took is
asked of the engine."""
import ctypes as C

import numpy as np
import pytest

from tests.test_gpu_engine import small_cfg
from tests.test_gpu_stack import config_a
from vllm_rs_amd import checkpoint
from vllm_rs_amd.engine import Engine

pytestmark = pytest.mark.gpu


def stack(dtype):
    cj = config_a()
    cj.update(width=96, vocab=1000)
    return checkpoint.parse_config(cj, dtype)


FORMS = {"llama": (lambda: small_cfg(vocab_size=8192), (1, 2, 3, 4, 5, 16, 17, 32, 33, 40)), "llama wide": (lambda: small_cfg(hidden_size=4096, num_layers=1, vocab_size=4112), (1, 3, 4, 15, 17, 32)),
         "stack": (lambda: stack(None), (1, 8, 9, 17, 32, 33)), "stack f32": (lambda: stack("float32"), (1, 17))}


@pytest.mark.parametrize("form", FORMS)
def test_pinned_rows_are_those_of_the_copy(form):
    make, sizes = FORMS[form]
    eng = Engine(make(), num_gpu_blocks=48, max_num_seqs=40, max_model_len=128, use_graph=False).init_synthetic()
    L, V = eng.L, eng.mc.vocab_size
    room = 41 * V * 4
    ptr = L.vra_malloc_host(room)
    pinned = np.ctypeslib.as_array((C.c_uint32 * (room // 4)).from_address(ptr))
    r = np.random.default_rng(len(form))

    def step(B, at, prompt):
        a = [r2.integers(0, V, B).astype(np.uint32), np.zeros(B, np.int64), np.arange(B, dtype=np.int64) * 64, np.arange(B, dtype=np.uint32).reshape(B, 1), np.ones(B, np.uint32)]
        cu = np.arange(B + 1, dtype=np.uint32) if prompt else None
        p = [v.ctypes.data_as(C.c_void_p) for v in a]
        rc = L.vra_engine_forward_raw(eng.h, p[0], p[1], p[2], B, int(prompt), p[3], 1, p[4], cu.ctypes.data_as(C.c_void_p) if prompt else None, B, C.c_void_p(at))
        eng._check(rc, "forward_raw")

    try:
        for B in sizes:
            for prompt in (False, True):
                n, seed = B * V, int(r.integers(1 << 30))
                plain = np.full(n + 2, 0xABABABAB, np.uint32)
                r2 = np.random.default_rng(seed)
                step(B, plain.ctypes.data + 4, prompt)
                assert not L.vra_engine_logits_in_place(eng.h)
                assert plain[0] == plain[-1] == 0xABABABAB and np.isfinite(plain[1:-1].view(np.float32)).all() and plain[1:-1].any()
                for start in (room // 4 - n, 16, 15):  # to the last byte, in the middle, off 16 bytes
                    pinned[:] = 0xCDCDCDCD
                    r2 = np.random.default_rng(seed)
                    step(B, ptr + start * 4, prompt)
                    assert L.vra_engine_logits_in_place(eng.h) == (start % 4 == 0 and B <= 32 and form != "stack f32"), (B, prompt, start)
                    assert np.array_equal(pinned[start:start + n], plain[1:-1]), (B, prompt, start)
                    assert (pinned[:start] == 0xCDCDCDCD).all() and (pinned[start + n:] == 0xCDCDCDCD).all()
                    kept = np.empty(n, np.uint32)  # (the device's rows are there as before)
                    assert L.vra_engine_copy_logits(eng.h, kept.ctypes.data_as(C.c_void_p), B) == 0 and np.array_equal(kept, plain[1:-1])
    finally:
        del pinned
        L.vra_free_host(ptr)
        eng.close()
