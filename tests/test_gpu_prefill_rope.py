"""Prompt attention that rotates the queries as it reads them (vra_rope_cache_attention_prefill): the bits of the launches one by one, in the result and in the cache."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.util import BF16, F16, rand_dt, rng
from vllm_rs_amd import ops

pytestmark = pytest.mark.gpu


# 64 and 128 rows a workgroup (many heads), ragged last blocks, rows behind a cached prefix (positions from the middle), both caches; a window: the general kernel
@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("Hq,Hkv,D,new,old,window", [(32, 8, 128, [5, 70, 1], [0, 33, 200], 0), (7, 1, 64, [129, 64], [0, 100], 0), (32, 4, 64, [1100, 131], [0, 64], 0),
                                                     (28, 4, 128, [1030, 257, 300], [0, 0, 90], 0), (8, 2, 128, [40, 90], [0, 50], 48)])
def test_same_bits_as_one_by_one(Hq, Hkv, D, new, old, window, fp8, dt):
    L, BS, B, T = ops.lib(), 64, len(new), sum(new)
    r = rng(T + D + Hq + fp8 + dt)
    ctx = [n + o for n, o in zip(new, old)]
    mb = max((c + BS - 1) // BS for c in ctx)
    NB = B * mb
    bt = r.permutation(NB).reshape(B, mb).astype(np.uint32)
    slots = np.array([int(bt[b, j // BS]) * BS + j % BS for b in range(B) for j in range(old[b], ctx[b])], np.int64)
    pos = np.concatenate([np.arange(o, c) for o, c in zip(old, ctx)]).astype(np.int64)
    cos, sin = (orc.to_dt(t, dt) for t in orc.rope_tables(D, 10000.0, 2048))
    q, k, v = rand_dt(r, (T, Hq, D), dt), rand_dt(r, (T, Hkv, D), dt), rand_dt(r, (T, Hkv, D), dt)
    es, kvdt = (1, 3) if fp8 else (2, dt)
    history = r.integers(0, 64, NB * Hkv * BS * D * es).astype(np.uint8)  # (finite in every type)
    common = [ops.dev(a) for a in (cos, sin, pos, slots, bt, np.array(ctx, np.uint32), np.concatenate([[0], np.cumsum(new)]).astype(np.uint32))]
    c, s, p, sl, tab, cl, cu = (d.ptr for d in common)

    def run(fused):
        dq, dk, dv, kc, vc = ops.dev(q), ops.dev(k), ops.dev(v), ops.dev(history), ops.dev(history)
        out = ops.DevBuf(T * Hq * D * 2).fill_bytes(0)
        if fused:
            L.vra_rope_cache_attention_prefill(out.ptr, dq.ptr, dk.ptr, dv.ptr, kc.ptr, vc.ptr, c, s, p, sl, tab, cl, cu, B, T, max(new), Hq, Hkv, D, BS, mb, D ** -0.5,
                                               window, dt, kvdt, 0)
        else:
            L.vra_rope_cache_prefill(dq.ptr, dk.ptr, dv.ptr, kc.ptr, vc.ptr, c, s, p, sl, T, Hq, Hkv, D, BS, dt, kvdt, 0)
            L.vra_paged_attention_prefill_sw(out.ptr, dq.ptr, None, None, kc.ptr, vc.ptr, tab, cl, cu, None, B, T, max(new), Hq, Hkv, D, BS, mb, D ** -0.5, 0.0, window, dt,
                                             kvdt, 0)
        ops.check_error()
        return out.numpy(np.uint16, (T, Hq, D)), kc.numpy(np.uint8, history.shape), vc.numpy(np.uint8, history.shape)
    got, ref = run(True), run(False)
    assert ref[0].any() and all(np.array_equal(a, b) for a, b in zip(got, ref))
