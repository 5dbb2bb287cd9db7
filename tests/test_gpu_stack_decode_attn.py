"""The decode attention of layer stacks with a key/value head's query heads together and the context in parts, against softmax attention in
float64: part and tile edges (128 and 16 keys), one key, more keys than `splits` parts of 128, no key at all, 32 parts; 1..8 query heads a key/value head;
pages of 8 to 128 keys; head sizes of every template and between them; cap, temperature, block mask, window, sink, scale and gate per head; three launches on one scratch.

The weights and sums are float32 and the stored row is bf16: 2^-9 of a value, 4e-3 of the rows' norm."""
import math

import numpy as np
import pytest

from tests.test_gpu_stack import BF16, check, empty, from_dev, raw, rel, to_dev
from vllm_rs_amd import _lib, checkpoint

pytestmark = pytest.mark.gpu

b16 = lambda x: (checkpoint.f32_to_bf16_bits(np.ascontiguousarray(x, np.float32)).astype(np.uint32) << 16).view(np.float32)


def reference(q, k, v, p, scale, softcap, coef, every, chunk, window, sink, hs, gate):
    H, G = q.shape[0], k.shape[1]
    n = min(k.shape[0], p + 1)
    out = np.zeros((H, v.shape[2]))
    lo = p // chunk * chunk if chunk else 0
    if window:
        lo = max(lo, p - window + 1)
    for h in range(H):
        g = h // (H // G)
        s = (k[lo:n, g].astype(np.float64) @ q[h]) * scale * (hs[h] if hs is not None else 1.0)
        if every:
            s = s * (1.0 + coef * math.log((p + 1) // every + 1.0))
        if softcap:
            s = softcap * np.tanh(s / softcap)
        top = max([s.max()] if len(s) else [-np.inf] + ([sink[h]] if sink is not None else []))
        if not len(s) and sink is None:
            continue
        top = max(top, sink[h]) if sink is not None else top
        e = np.exp(s - top)
        o = e @ v[lo:n, g] / (e.sum() + (math.exp(sink[h] - top) if sink is not None else 0.0))
        out[h] = o / (1.0 + math.exp(-gate[h])) if gate is not None else o
    return out


def decode_in_parts(H, G, dim, vdim, splits, form, lens, BS):
    L = _lib.load()
    r = np.random.default_rng(dim + vdim + splits)
    B = len(lens)
    per = [max(1, (n + BS - 1) // BS) for n in lens]
    order = r.permutation(sum(per) + 2).astype(np.uint32)
    tables = np.zeros((B, max(per)), np.uint32)
    kc = np.full(((sum(per) + 2) * BS, G, dim), 1e4, np.float32)
    vc = np.full(((sum(per) + 2) * BS, G, vdim), -1e4, np.float32)
    ks, vs, at = [], [], 0
    for i, n in enumerate(lens):
        tables[i, :per[i]] = order[at:at + per[i]]
        at += per[i]
        k, v = b16(r.standard_normal((n, G, dim))), b16(r.standard_normal((n, G, vdim)))
        slots = tables[i, np.arange(n) // BS].astype(np.int64) * BS + np.arange(n) % BS
        kc[slots], vc[slots] = k, v
        ks.append(k), vs.append(v)
    q = b16(r.standard_normal((B, H, dim)) * 1.5)
    pos = np.array([max(n - 1, 0) for n in lens], np.int64)
    scale, softcap, coef, every, chunk, window, sink, hs, gate = dim ** -0.5, 0.0, 0.0, 0, 0, 0, None, None, None
    if form == "capped":
        softcap, coef, every = 2.0, 0.1, 100
    elif form == "block":
        chunk = 70
    elif form == "window":
        window = 150
    elif form == "dressed":
        sink, hs, gate = r.standard_normal(H).astype(np.float32), (0.5 + r.random(H)).astype(np.float32), r.standard_normal((B, H)).astype(np.float32)
    R = 1 << max(0, (H // G - 1).bit_length())
    W = 64 if max(dim, vdim) <= 64 else 128 if max(dim, vdim) <= 128 else 256
    nbytes = B * G * splits * R * (W + 2) * 4
    scratch, arrived = empty(nbytes), raw(np.zeros(B * G), np.uint32)
    dp = lambda a: raw(a, np.float32).ptr if a is not None else None
    args = (to_dev(q, BF16).ptr, H * dim)
    rest = (to_dev(kc, BF16).ptr, to_dev(vc, BF16).ptr, raw(pos, np.int64).ptr, raw(tables, np.uint32).ptr, raw(lens, np.uint32).ptr, B, H, G, dim, vdim, BS,
            tables.shape[1], scale, softcap, coef, every, chunk, window, dp(sink), dp(hs), dp(gate), H)
    got = []
    for parts in (True, True, True, False):  # the last one without scratch: the one-head kernel
        out = empty(B * H * vdim * 2)
        L.vra_stack_op_attention_decode(*args, out.ptr, *rest, scratch.ptr if parts else None, nbytes if parts else 0, splits if parts else 0,
                                        arrived.ptr if parts else None, BF16, 0)
        check()
        got.append(from_dev(out, (B, H, vdim), BF16))
    assert (got[0] == got[1]).all() and (got[0] == got[2]).all() and not arrived.numpy(np.uint32, (B * G,)).any()
    for i in range(B):
        ref = reference(q[i], ks[i], vs[i], int(pos[i]), scale, softcap, coef, every, chunk, window, sink, hs, gate[i] if gate is not None else None)
        for a in (got[0], got[3]):
            assert rel(a[i], ref) < 4e-3 if ref.any() else not a[i].any(), (lens[i], rel(a[i], ref))


@pytest.mark.parametrize("form", ["plain", "capped", "block", "window", "dressed"])
@pytest.mark.parametrize("H,G,dim,vdim,splits", [(16, 4, 128, 128, 8), (8, 8, 64, 64, 8), (16, 2, 72, 40, 3), (4, 2, 256, 200, 2), (6, 2, 24, 136, 32), (8, 1, 128, 128, 1)])
def test_decode_attention_in_parts(H, G, dim, vdim, splits, form):
    decode_in_parts(H, G, dim, vdim, splits, form, [1, 31, 32, 33, 127, 128, 129, 300, 1100, 0], 64)


@pytest.mark.parametrize("form", ["plain", "capped", "dressed"])
@pytest.mark.parametrize("H,G,dim,vdim", [(8, 4, 64, 64), (16, 4, 128, 128), (8, 2, 256, 256), (8, 1, 256, 200)])
def test_long_contexts_fill_the_parts(H, G, dim, vdim, form):
    """17 and 32 parts of 128 keys, 18 of 256: the upper half of the lanes that weigh the parts, all four rounds of their rows"""
    decode_in_parts(H, G, dim, vdim, 32, form, [2049, 4096, 4500, 130], 64)


@pytest.mark.parametrize("BS", [8, 24, 100, 128])
@pytest.mark.parametrize("H,G,dim,vdim,splits,form", [(16, 4, 128, 128, 8, "plain"), (8, 8, 64, 64, 2, "block"), (16, 2, 72, 40, 3, "dressed"), (4, 2, 256, 200, 4, "window")])
def test_pages_that_a_wave_crosses(H, G, dim, vdim, splits, form, BS):
    """pages smaller than a wave's 16 keys or off them: lanes of one load lie in several pages, and the page asked for ahead is some lanes' only"""
    decode_in_parts(H, G, dim, vdim, splits, form, [1, BS - 1, BS, BS + 1, 127, 129, 333, 1100, 0], BS)
