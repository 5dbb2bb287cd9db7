"""Prompt attention (csrc/attn_prefill.cuh) rescales the outputs of a row tile only where a maximum of it moved: scores that climb by little and by much
from tile to tile, that jump, and that fall; against the softmax in float64.

p is rounded to 16 bits on its way into p . v and the output once more, each by at most half a unit in the last place (2^-8 of the value in bf16's
8 bits, 2^-11 in f16's 11); the sum of the p is not: 2^-7 (2^-10) of sum_j p_j |v_j| / sum_j p_j, and f32 sums below a twentieth of that."""
import numpy as np
import pytest

from oracle import oracle as orc
from tests.test_gpu_kernels import _paged_setup
from tests.util import BF16, F16, rng
from vllm_rs_amd import ops

pytestmark = pytest.mark.gpu

CTX = 330
KEYS = np.arange(CTX)
PROFILES = {  # score of key j, log2
    "climbs a little": KEYS * (7.5 / CTX),
    "climbs": KEYS * 0.11,
    "a step a tile": 8.0 * (KEYS // 64),
    "jumps": np.where(KEYS % 100 == 99, 40.0, 0.0) + (KEYS // 100) * 30.0,
    "falls": 60.0 - KEYS * 0.3,
    "one key far above": np.where(KEYS == 70, 90.0, -20.0),
}


@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("prefix", [0, 70])
@pytest.mark.parametrize("profile", list(PROFILES))
def test_rows_whose_maxima_move(profile, prefix, D, dt):
    r = rng(D + prefix + len(profile))
    Hq, Hkv, BS, lq = 4, 2, 64, CTX - prefix
    s = _paged_setup(r, [CTX], Hkv, D, BS, dt)
    scale = D ** -0.5
    q = orc.to_dt((r.standard_normal((lq, Hq, D)) * 0.05).astype(np.float32), dt)
    qf = orc.from_dt(q, dt).copy()
    qf[:, :, 0] = 8.0
    kf = (r.standard_normal((CTX, Hkv, D)) * 0.05).astype(np.float32)
    kf[:, :, 0] = (PROFILES[profile] * np.log(2.0) / (8.0 * scale))[:, None]
    q, k = orc.to_dt(qf, dt), orc.to_dt(kf, dt)
    qf, kf, vf = (orc.from_dt(t, dt).astype(np.float64) for t in (q, k, s["v"]))
    pa = ops.PagedAttention(Hq, D, scale, Hkv, BS, dt)
    pa.reshape_and_cache(ops.dev(k), ops.dev(s["v"]), s["kc"], s["vc"], ops.dev(s["slots"]), len(s["slots"]))
    out = pa.forward_prefill(ops.dev(q), lq, lq, ops.dev(np.array([0, lq], np.uint32)), 1, k_cache=s["kc"], v_cache=s["vc"], block_tables=ops.dev(s["bt"]),
                             context_lens=ops.dev(np.array([CTX], np.uint32)), max_blocks=s["max_blocks"])
    got = orc.from_dt(out.numpy(np.uint16, (lq, Hq, D)), dt).astype(np.float64)
    unit = 2.0 ** -7 if dt == BF16 else 2.0 ** -10
    for h in range(Hq):
        z = qf[:, h] @ kf[:, h * Hkv // Hq].T * scale
        z[KEYS[None, :] > (prefix + np.arange(lq))[:, None]] = -np.inf
        p = np.exp(z - z.max(1, keepdims=True))
        v = vf[:, h * Hkv // Hq]
        ref, mag = p @ v / p.sum(1, keepdims=True), p @ np.abs(v) / p.sum(1, keepdims=True)
        assert (np.abs(got[:, h] - ref) <= 1.05 * unit * mag + 1e-6).all(), (h, float((np.abs(got[:, h] - ref) / (unit * mag)).max()))


@pytest.mark.parametrize("dt", [BF16, F16])
@pytest.mark.parametrize("D", [64, 128])
@pytest.mark.parametrize("ctxs,prefix", [([1, 33], 0), ([330, 97], 70), ([700], 0)])
def test_block_sizes_and_the_fp8_cache(ctxs, prefix, D, dt):
    """where a key or value lies changes no bit, nor does a cache of 8 bits whose numbers hold the values exactly"""
    r = rng(D + sum(ctxs) + dt)
    Hq, Hkv = 8, 2
    lq = [c - min(prefix, c - 1) for c in ctxs]
    k, v = (orc.to_dt((r.integers(-7, 8, (sum(ctxs), Hkv, D)) / 4.0).astype(np.float32), dt) for _ in range(2))  # (three bits behind the point)
    q = orc.to_dt(r.standard_normal((sum(lq), Hq, D)).astype(np.float32), dt)
    outs = []
    for BS in (64, 32, 128):
        for fp8 in (False, True):
            need = [-(-c // BS) for c in ctxs]
            perm = r.permutation(sum(need) + 2).astype(np.uint32)
            bt = np.zeros((len(ctxs), max(need)), np.uint32)
            for b, n in enumerate(need):
                bt[b, :n] = perm[sum(need[:b]):sum(need[:b + 1])]
            slots = np.concatenate([bt[b, np.arange(c) // BS].astype(np.int64) * BS + np.arange(c) % BS for b, c in enumerate(ctxs)])
            bytes_ = (sum(need) + 2) * BS * Hkv * D * (1 if fp8 else 2)
            kc, vc = (ops.DevBuf(bytes_).fill_bytes(0x7F if fp8 else 0xFF) for _ in range(2))  # (NaN)
            pa = ops.PagedAttention(Hq, D, D ** -0.5, Hkv, BS, dt, fp8_kvcache=fp8)
            pa.reshape_and_cache(ops.dev(k), ops.dev(v), kc, vc, ops.dev(slots), len(slots))
            out = pa.forward_prefill(ops.dev(q), sum(lq), max(lq), ops.dev(np.concatenate([[0], np.cumsum(lq)]).astype(np.uint32)), len(ctxs), k_cache=kc, v_cache=vc,
                                     block_tables=ops.dev(bt), context_lens=ops.dev(np.array(ctxs, np.uint32)), max_blocks=max(need))
            outs.append(out.numpy(np.uint16, (sum(lq), Hq, D)))
    assert np.isfinite(orc.from_dt(outs[0], dt)).all() and outs[0].any()
    assert all(np.array_equal(o, outs[0]) for o in outs[1:])
