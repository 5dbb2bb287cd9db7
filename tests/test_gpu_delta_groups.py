"""The gated delta rule over prompts of few columns, in three groups of waves (rows off 16 bytes: in one), against the float64 recurrence: lengths around the
edges of the tiles of 8 tokens, ragged batches with an empty slot, key sizes of both templates, value sizes off a workgroup's columns, grouped
q / k heads, rows apart, one decay a head, decays of 0 and 1, a state that waits between portions.

float32 sums of 64..128 terms along chains that contract (decays up to 1, unit keys, write strengths up to 1): 1e-5 of the largest output."""
import numpy as np
import pytest

from tests import zifetar_oracle as zo
from tests.test_gpu_stack import check, empty, raw
from vllm_rs_amd import _lib

pytestmark = pytest.mark.gpu


def worst(got, ref):
    return float(np.abs(got - ref).max() / np.abs(ref).max())


@pytest.mark.parametrize("lens", [[1], [2, 7, 8], [9, 1, 17, 31], [100, 48, 64, 49, 5]], ids=str)
@pytest.mark.parametrize("per_head", [False, True], ids=["channels", "heads"])
@pytest.mark.parametrize("D,V,H,rep,pad", [(64, 20, 2, 1, 0), (64, 64, 4, 2, 4), (128, 128, 2, 2, 0), (128, 45, 3, 1, 0), (128, 24, 2, 1, 1)])
def test_delta_rule_in_groups(D, V, H, rep, pad, per_head, lens):
    L = _lib.load()
    r = np.random.default_rng(D + V + sum(lens) + per_head)
    B, T = len(lens), sum(lens)
    q, k = (r.standard_normal((T, H // rep, D)).astype(np.float32) for _ in "qk")
    k /= np.sqrt((k * k).sum(-1, keepdims=True))
    v = r.standard_normal((T, H, V)).astype(np.float32)
    decay = (0.5 + 0.5 * r.random((T, H) if per_head else (T, H, D))).astype(np.float32)
    decay[r.random(decay.shape) < 0.05] = 0.0
    decay[r.random(decay.shape) < 0.2] = 1.0
    beta = r.random((T, H)).astype(np.float32)
    skipped = B - 1 if B > 2 else None  # a sequence without a slot: its rows of the output stay as they are

    def rows(x):
        x = x.reshape(len(x), -1)
        y = np.full((len(x), x.shape[1] + pad), 9.0, np.float32)
        y[:, :x.shape[1]] = x
        return raw(y, np.float32).ptr

    state = raw(np.full((B + 1) * H * V * D, 50.0, np.float32), np.float32)  # (what earlier sequences left)
    slots = np.arange(B, dtype=np.int32) + 1
    if skipped is not None:
        slots[skipped] = -1
    starts = np.concatenate([[0], np.cumsum(lens)])

    def run(parts):  # parts: rows (first, last) of every sequence
        idx = np.concatenate([np.arange(starts[i] + a, starts[i] + b) for i, (a, b) in enumerate(parts)])
        cu = np.concatenate([[0], np.cumsum([b - a for a, b in parts])])
        pos = np.concatenate([np.arange(a, b) for a, b in parts])
        out = empty(len(idx) * (H * V + pad) * 4)
        L.vra_stack_op_linear_scan_ex(rows(q[idx]), H // rep * D + pad, rows(k[idx]), H // rep * D + pad, rows(v[idx]), H * V + pad, rows(decay[idx]),
                                      (H if per_head else H * D) + pad, int(per_head), 0, None, rows(beta[idx]), H + pad, 0.5, state.ptr,
                                      raw(slots, np.int32).ptr, raw(pos, np.int64).ptr, raw(cu, np.uint32).ptr, out.ptr, H * V + pad, B, H, rep, D, V, 0)
        check()
        o = out.numpy(np.float32, (len(idx), H * V + pad))
        assert np.isnan(o[:, H * V:]).all()  # (nothing is written between the rows)
        return [o[cu[i]:cu[i + 1], :H * V].reshape(-1, H, V) for i in range(B)]

    whole = run([(0, n) for n in lens])
    s1 = state.numpy(np.float32, (B + 1, H, V, D)).copy()
    half = [max(1, n // 2) if n > 1 else 1 for n in lens]
    first = run([(0, c) for c in half])
    second = run([(c, n) for c, n in zip(half, lens)]) if all(c < n for c, n in zip(half, lens)) else None
    s2 = state.numpy(np.float32, (B + 1, H, V, D))
    assert (s1[0] == 50.0).all()
    for i, n in enumerate(lens):
        at = slice(starts[i], starts[i] + n)
        if i == skipped:
            assert np.isnan(whole[i]).all()
            continue
        dd = np.broadcast_to(decay[at][:, :, None], (n, H, D)) if per_head else decay[at]
        ref = zo.linear_recurrence(np.repeat(q[at], rep, 1).astype(np.float64) * 0.5, np.repeat(k[at], rep, 1).astype(np.float64), v[at].astype(np.float64),
                                   dd.astype(np.float64), beta[at].astype(np.float64))
        S = np.zeros((H, V, D))
        for t in range(starts[i], starts[i] + n):
            S = S * (decay[t][:, None, None] if per_head else decay[t][:, None, :]).astype(np.float64)
            kk = np.repeat(k[t], rep, 0).astype(np.float64)
            u = beta[t][:, None] * (v[t] - (S * kk[:, None, :]).sum(-1))
            S = S + u[:, :, None] * kk[:, None, :]
        assert worst(whole[i], ref) < 1e-5 and worst(s1[slots[i]], S) < 1e-5, (n, worst(whole[i], ref), worst(s1[slots[i]], S))
        assert worst(first[i], ref[:half[i]]) < 1e-5
        if second is not None:
            assert worst(second[i], ref[half[i]:]) < 1e-5 and worst(s2[slots[i]], S) < 1e-5
