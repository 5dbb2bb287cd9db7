"""Decode attention over the FP8 cache (decode_attn_fused_kernel): waves with one to eight tiles of 32 tokens, whose loop requests a tile ahead, against the oracle."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.util import BF16, F16, assert_close_dt, rand_dt, rng
from vllm_rs_amd import ops

pytestmark = pytest.mark.gpu


# without a workspace one workgroup (four waves) takes the whole context: 1 .. 8 tiles a wave, waves with one tile more than others, a last tile of one token
@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("Hq,Hkv,D", [(8, 2, 128), (7, 1, 64)])
@pytest.mark.parametrize("ctxs", [[257, 384], [385, 480], [512, 513], [640, 700], [768, 801], [897, 1024]])
def test_tiles_of_a_wave(ctxs, Hq, Hkv, D, dt):
    BS, NB, B = 64, 64, len(ctxs)
    r = rng(sum(ctxs) + D + dt)
    mb = max((c + BS - 1) // BS for c in ctxs)
    bt = r.permutation(NB)[:B * mb].reshape(B, mb).astype(np.uint32)
    slot = lambda b, j: int(bt[b, j // BS]) * BS + j % BS
    hs = np.array([slot(b, j) for b, c in enumerate(ctxs) for j in range(c - 1)], np.int64)
    hk, hv = rand_dt(r, (len(hs), Hkv, D), dt, 2.0), rand_dt(r, (len(hs), Hkv, D), dt, 2.0)
    kr_, vr_ = np.zeros((NB, Hkv, BS, D), np.uint8), np.zeros((NB, Hkv, D, BS), np.uint8)
    kc, vc = ops.DevBuf(kr_.nbytes).fill_bytes(0x7F), ops.DevBuf(vr_.nbytes).fill_bytes(0x7F)  # (NaN)
    pa = ops.PagedAttention(Hq, D, D ** -0.5, Hkv, BS, dt, fp8_kvcache=True)
    orc.reshape_and_cache(hk, hv, kr_, vr_, hs, BS, dt, orc.FP8)
    pa.reshape_and_cache(ops.dev(hk), ops.dev(hv), kc, vc, ops.dev(hs), len(hs))
    q, k, v = rand_dt(r, (B, Hq, D), dt), rand_dt(r, (B, Hkv, D), dt, 2.0), rand_dt(r, (B, Hkv, D), dt, 2.0)
    pos, slots = np.array(ctxs, np.int64) - 1, np.array([slot(b, c - 1) for b, c in enumerate(ctxs)], np.int64)
    cos, sin = (orc.to_dt(t, dt) for t in orc.rope_tables(D, 10000.0, 2048))
    cl = np.array(ctxs, np.uint32)
    qr, kr = orc.rope(q, cos, sin, pos, False, dt, dt), orc.rope(k, cos, sin, pos, False, dt, dt)
    orc.reshape_and_cache(kr, v, kr_, vr_, slots, BS, dt, orc.FP8)
    ref = orc.paged_attention(qr, kr_, vr_, bt, cl, None, Hkv, BS, D ** -0.5, dt, kv_dt=orc.FP8)
    out = pa.rope_cache_decode(ops.dev(q), ops.dev(k), ops.dev(v), kc, vc, ops.dev(cos), ops.dev(sin), ops.dev(pos), ops.dev(slots), ops.dev(bt), ops.dev(cl), B, mb,
                               max(ctxs), None)
    # (two storage ulps as in the other decode tests: the rotated q and k may each round to the neighbour, an E4M3 step of one key in hundreds)
    assert_close_dt(out.numpy(np.uint16, (B, Hq, D)), ref, dt, max_ulp=2.0, max_mismatch_frac=0.5, name="fp8 decode tiles", abs_floor=8e-3 if dt == BF16 else 1.5e-3)


# many sequences: waves that load a tile, then compute it (three tiles on a full chip, heads of 64 beyond three workgroups a CU, heads of 128 in one round of two), against the same
# sequences by threes, whose waves request a tile ahead: the same bits
@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("B,Hq,Hkv,D,ctxs", [(33, 16, 8, 128, [384, 257, 33, 1]), (33, 8, 8, 128, [1024, 641, 96, 130]), (33, 8, 8, 64, [384, 290, 5, 32]),
                                             (98, 32, 8, 64, [700, 1, 129, 544])])
def test_many_sequences_have_the_bits_of_few(B, Hq, Hkv, D, ctxs, dt):
    BS = 64
    r = rng(B + D + ctxs[0])
    mb, ctx = (max(ctxs) + BS - 1) // BS, np.array([ctxs[b % len(ctxs)] for b in range(B)], np.uint32)
    bt = r.permutation(B * mb).reshape(B, mb).astype(np.uint32)
    kc, vc = (ops.dev(r.integers(0, 0x78, (B * mb, Hkv, BS * D // 4, 4), np.uint8).view(np.uint32)) for _ in range(2))
    q, k, v = rand_dt(r, (B, Hq, D), dt), rand_dt(r, (B, Hkv, D), dt, 2.0), rand_dt(r, (B, Hkv, D), dt, 2.0)
    pos = ctx.astype(np.int64) - 1
    slots = bt[np.arange(B), pos // BS].astype(np.int64) * BS + pos % BS
    cos, sin = (ops.dev(orc.to_dt(t, dt)) for t in orc.rope_tables(D, 10000.0, 2048))
    pa = ops.PagedAttention(Hq, D, D ** -0.5, Hkv, BS, dt, fp8_kvcache=True)

    def run(b):
        out = pa.rope_cache_decode(ops.dev(q[b]), ops.dev(k[b]), ops.dev(v[b]), kc, vc, cos, sin, ops.dev(pos[b]), ops.dev(slots[b]), ops.dev(bt[b]), ops.dev(ctx[b]), len(q[b]), mb,
                                   int(ctx.max()), None)
        return out.numpy(np.uint16, (len(q[b]), Hq, D))

    many = run(slice(None))
    assert np.isfinite(orc.from_dt(many, dt)).all() and many.any()
    for b in range(0, B, 3):
        assert np.array_equal(run(slice(b, b + 3)), many[b:b + 3]), b
