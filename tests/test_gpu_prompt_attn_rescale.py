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
