"""The tile kernel of prompt steps takes each 64-key tile in two halves of 32 keys, joined at the end (csrc/stack_prompt_attn.hip): against float64 where a
half holds no key, one, or none that a row sees; rows of a page's end; scores far beyond the cap, of either sign.  And the rows of a prompt cut in portions are
the whole prompt's, bit for bit.

bf16: the output's rounding, 2^-9 of a value, and a weight's tail at 2^-17."""
import numpy as np
import pytest

from tests.test_gpu_stack import BF16, check, empty, from_dev, paged, raw, rel, to_dev
from tests import stack_oracle as so
from vllm_rs_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim,vdim", [(64, 64), (128, 128), (64, 128), (128, 64)])
@pytest.mark.parametrize("cap,scale", [(0.0, 0.1), (5.0, 0.1), (5.0, 40.0), (5.0, -0.1)])
@pytest.mark.parametrize("first,Tq,window", [(0, 31, 0), (0, 32, 0), (0, 33, 0), (96, 97, 0), (31, 130, 16), (64, 65, 33), (127, 1, 1)])
def test_halves_of_a_tile(dim, vdim, cap, scale, first, Tq, window):
    if cap and window:
        pytest.skip("no entry point takes a cap and a window")
    L = _lib.load()
    r = np.random.default_rng(dim + vdim + first + Tq)
    H, G, Tk = 4, 2, first + Tq
    k, v, q = (so.bf16_round(r.standard_normal(s).astype(np.float32)) for s in ((Tk, G, dim), (Tk, G, vdim), (Tq, H, dim)))
    kc, vc, table = paged(k, v, 64, r, BF16)

    def run(a, b):
        n = b - a
        out = empty(n * H * vdim * 2)
        args = (to_dev(q[a:b].reshape(n, -1), BF16).ptr, H * dim, out.ptr, kc.ptr, vc.ptr, raw(np.arange(first + a, first + b), np.int64).ptr,
                raw(table, np.uint32).ptr, raw([first + b], np.uint32).ptr, raw([0, n], np.uint32).ptr, 1, n, n, H, G, dim, vdim, 64, len(table), scale)
        if window:
            L.vra_stack_op_attention_window(*args, window, None, None, None, H, BF16, 0)
        else:
            L.vra_stack_op_attention(*args, cap, 0.0, 0, BF16, 0)
        check()
        return from_dev(out, (n, H, vdim), BF16)

    p, j = np.arange(first, Tk)[:, None], np.arange(Tk)[None]
    ref = np.zeros((Tq, H, vdim))
    for h in range(H):
        s = q[:, h].astype(np.float64) @ k[:, h // 2].astype(np.float64).T * scale
        s = cap * np.tanh(s / cap) if cap else s
        s = np.where((j <= p) & (j > p - window if window else True), s, -np.inf)
        e = np.exp(s - s.max(-1, keepdims=True))
        ref[:, h] = e / e.sum(-1, keepdims=True) @ v[:, h // 2].astype(np.float64)
    got = run(0, Tq)
    assert rel(got, ref) < 4e-3
    for a, b in ((0, Tq // 3), (Tq // 3, Tq)):
        if b > a:
            assert (run(a, b) == got[a:b]).all()
