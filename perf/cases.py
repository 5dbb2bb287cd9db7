"""What this framework is used for, as measurable cases.

Whole models run through `vllm_rs_amd.engine.Engine`: weights in checkpoint format are loaded once, and one pass is one forward step
(`forward_raw`) of a batch behind its paged cache, logits out.  The int4 decoders (GPTQ and AWQ, the widths of engine.py's tables), the
dense bf16 / f16 decoder and the layer-stack decoder (Ditilix) are covered in prompt steps and in decode steps, from one token to
thousands, with ragged batches, both 16-bit types and the FP8 cache.  The two attention-like operators of the recurrent and latent
designs are called through the C ABI as a host program calls them, on caller-owned device buffers.

Models are cut to a few layers and a 32 000-token vocabulary: every layer is the same work, and a step's time is the sum over them.
"""
import math

import numpy as np
import torch

from vllm_rs_amd import _lib
from vllm_rs_amd import engine as eng_mod

VOCAB = 32000
BS = 64  # tokens of a cache block

LLAMA = {"llama3-8b": eng_mod.LLAMA3_8B, "qwen2-7b": eng_mod.QWEN2_7B, "llama3-70b-tp8-rank": eng_mod.LLAMA3_70B_TP8_RANK, "tinyllama": eng_mod.TINYLLAMA}
STACK = {  # width, heads, kv heads, head size, dense feed-forward, experts, chosen, expert size, shared expert
    "dense-2048": (2048, 16, 4, 128, 8192, 0, 0, 0, 0),
    "moe-2048": (2048, 16, 4, 128, 8192, 16, 2, 1024, 2048),
    "dense-4096": (4096, 32, 8, 128, 14336, 0, 0, 0, 0),
}


def listed():
    return [
        # one user's chat turn: a single sequence decodes behind a short context (the headline workload's step)
        dict(name="int4 decode 1", kind="llama", model="llama3-8b", quant="gptq", dtype="bf16", layers=4, phase="decode", seqs=1, tokens=500, fp8=False),
        # a serving batch: sixteen sequences of different lengths, AWQ weights with biases
        dict(name="int4 decode 16", kind="llama", model="qwen2-7b", quant="awq", dtype="bf16", layers=4, phase="decode", seqs=16, tokens=1900, fp8=False),
        # long documents behind an FP8 cache: the cache is most of the traffic
        dict(name="int4 decode 4 long fp8", kind="llama", model="llama3-8b", quant="gptq", dtype="bf16", layers=3, phase="decode", seqs=4, tokens=9001, fp8=True),
        # time to first token of a short question, f16 checkpoint
        dict(name="int4 prompt 150", kind="llama", model="llama3-8b", quant="gptq", dtype="f16", layers=4, phase="prompt", seqs=1, tokens=150, fp8=False),
        # a step that takes in three prompts of different lengths
        dict(name="int4 prompts 3x1021", kind="llama", model="qwen2-7b", quant="awq", dtype="bf16", layers=2, phase="prompt", seqs=3, tokens=1021, fp8=False),
        # one chunk of a long prompt (the default chunk size)
        dict(name="int4 prompt 8192", kind="llama", model="llama3-8b", quant="gptq", dtype="bf16", layers=2, phase="prompt", seqs=1, tokens=8192, fp8=False),
        # an unquantised small model taking in a batch of prompts
        dict(name="dense prompts 4x700", kind="llama", model="tinyllama", quant="none", dtype="bf16", layers=6, phase="prompt", seqs=4, tokens=700, fp8=False),
        # a layer-stack model: one prompt; and its mixture of experts
        dict(name="stack prompt 2048", kind="stack", model="dense-2048", dtype="bf16", layers=4, phase="prompt", seqs=1, tokens=2048),
        dict(name="stack experts prompt 1500", kind="stack", model="moe-2048", dtype="bf16", layers=3, phase="prompt", seqs=1, tokens=1500),
        # ... and a decode step of eight sequences behind chat-sized contexts
        dict(name="stack decode 8", kind="stack", model="dense-2048", dtype="bf16", layers=4, phase="decode", seqs=8, tokens=700),
        # the recurrence of a gated delta rule over a prompt (16 heads of 128), and latent attention of a decode batch (16 heads, rows of 512 + 64)
        dict(name="delta rule prompt 2048", kind="scan", heads=16, rep=4, dim=128, seqs=1, tokens=2048),
        dict(name="latent decode 8", kind="latent", heads=16, rank=512, rot=64, seqs=8, tokens=3900),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["llama"] * 6 + ["stack"] * 4 + ["scan", "latent"])
    if kind == "scan":
        return dict(kind=kind, heads=rng.choice([4, 8, 16, 32]), rep=rng.choice([1, 2, 4]), dim=rng.choice([64, 128]), seqs=rng.randint(1, 4),
                    tokens=_log(rng, 40, 2048))
    if kind == "latent":
        return dict(kind=kind, heads=rng.choice([8, 16, 32]), rank=rng.choice([192, 512]), rot=64, seqs=rng.randint(1, 8), tokens=_log(rng, 100, 3900))
    phase = rng.choice(["prompt", "decode"])
    if phase == "prompt":
        seqs, tokens = rng.randint(1, 4), _log(rng, 5, 4000)
        seqs = min(seqs, max(1, 8000 // tokens))
    else:
        seqs, tokens = _log(rng, 1, 32), _log(rng, 20, 9000)
        seqs = min(seqs, max(1, 30000 // tokens))
    if kind == "stack":
        model = rng.choice(["dense-2048", "dense-2048", "moe-2048", "dense-4096"])
        f32 = rng.random() < 0.15
        if f32:  # (the f32 form serves checks and small models)
            model, tokens, seqs = "dense-2048", min(tokens, 200), min(seqs, 2)
        if phase == "decode":
            tokens, seqs = min(tokens, 3000), min(seqs, 8)
        else:
            tokens = min(tokens, 2500)
            seqs = min(seqs, max(1, 4000 // tokens))
        return dict(kind=kind, model=model, dtype="f32" if f32 else "bf16", layers=1 if f32 else 2, phase=phase, seqs=seqs, tokens=tokens)
    model = rng.choice(["llama3-8b", "llama3-8b", "qwen2-7b", "qwen2-7b", "llama3-70b-tp8-rank", "tinyllama"])
    quant = "none" if model == "tinyllama" else rng.choice(["gptq", "awq"])
    if model == "tinyllama":
        tokens = min(tokens, 2000)
    return dict(kind=kind, model=model, quant=quant, dtype=rng.choice(["bf16", "bf16", "bf16", "f16"]), layers=2, phase=phase, seqs=seqs, tokens=tokens,
                fp8=phase == "decode" and rng.random() < 0.25)


# ---------------------------------------------------------------------------------------------------------------- inputs
def _lens(case):
    """the sequences' lengths: the longest first, the others between a quarter of it and all of it"""
    return [max(1, int(case["tokens"] * (1.0 if i == 0 else 0.25 + 0.75 * ((i * 0.6180339887) % 1.0)))) for i in range(case["seqs"])]


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(0x5EED + 7919 * int(seed))


_TORCH = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}


def _normal(g, shape, std, dtype, mean=0.0):
    return (torch.randn(shape, generator=g, device="cuda") * std + mean).to(dtype)


def _host(t):
    """a tensor as the checkpoint's bytes: 16-bit floats as their bit patterns"""
    if t.dtype in (torch.bfloat16, torch.float16):
        return t.view(torch.int16).cpu().numpy().view(np.uint16)
    if t.dtype == torch.int32:
        return t.cpu().numpy().view(np.uint32)
    return t.cpu().numpy()


def _llama_cfg(case):
    cfg = dict(LLAMA[case["model"]], num_layers=case["layers"], vocab_size=VOCAB, quant_method=None if case["quant"] == "none" else case["quant"],
               dtype=eng_mod.F16 if case["dtype"] == "f16" else eng_mod.BF16)
    cfg["max_position_embeddings"] = max(2048, (case["tokens"] + 64) // 64 * 64)
    return cfg


def _llama_shapes(cfg):
    H, D = cfg["hidden_size"], cfg["head_dim"]
    q, kv, ff = cfg["num_heads"] * D, cfg["num_kv_heads"] * D, cfg["intermediate_size"]
    return {"self_attn.q_proj": (H, q), "self_attn.k_proj": (H, kv), "self_attn.v_proj": (H, kv), "self_attn.o_proj": (q, H),
            "mlp.gate_proj": (H, ff), "mlp.up_proj": (H, ff), "mlp.down_proj": (ff, H)}


def _llama_tensors(case, cfg, seed):
    """(name, device tensor) in checkpoint format: int4 codes uniform, zero points 8 (GPTQ) or around 8 (AWQ), scales that give
    projections of unit gain; dense weights normal"""
    g, dt = _gen(seed), _TORCH[case["dtype"]]
    H = cfg["hidden_size"]
    yield "model.embed_tokens.weight", _normal(g, (VOCAB, H), 1.0, dt)
    yield "lm_head.weight", _normal(g, (VOCAB, H), H ** -0.5, dt)
    yield "model.norm.weight", _normal(g, (H,), 0.1, dt, 1.0)
    for i in range(cfg["num_layers"]):
        p = "model.layers.%d." % i
        yield p + "input_layernorm.weight", _normal(g, (H,), 0.1, dt, 1.0)
        yield p + "post_attention_layernorm.weight", _normal(g, (H,), 0.1, dt, 1.0)
        for name, (K, N) in _llama_shapes(cfg).items():
            if case["quant"] == "none":
                yield p + name + ".weight", _normal(g, (N, K), K ** -0.5, dt)
            else:
                groups = K // cfg["group_size"]
                shape = (K // 8, N) if case["quant"] == "gptq" else (K, N // 8)
                yield p + name + ".qweight", torch.randint(-2 ** 31, 2 ** 31, shape, generator=g, device="cuda", dtype=torch.int64).to(torch.int32)
                yield p + name + ".scales", ((torch.rand((groups, N), generator=g, device="cuda") * 0.8 + 0.6) * (K ** -0.5 / 4.6)).to(dt)
                if case["quant"] == "gptq":
                    yield p + name + ".qzeros", torch.full((groups, N // 8), 0x77777777, device="cuda", dtype=torch.int32)
                else:
                    nib = torch.randint(7, 10, (groups, N // 8, 8), generator=g, device="cuda", dtype=torch.int64)
                    z = (nib << (4 * torch.arange(8, device="cuda"))).sum(-1)
                    yield p + name + ".qzeros", torch.where(z >= 2 ** 31, z - 2 ** 32, z).to(torch.int32)
            if cfg.get("attention_bias") and name[10:11] in "qkv" and name.startswith("self_attn"):
                yield p + name + ".bias", _normal(g, (N,), 0.1, dt)


def _stack_json(case):
    W, heads, kvh, dim, ff, experts, top, eff, sff = STACK[case["model"]]
    layers = []
    for i in range(case["layers"]):
        mx = dict(heads=heads, kv_heads=kvh, dim=dim, vdim=dim, scale=dim ** -0.5, softcap=50.0, q_temp=dict(coef=0.1, every=1024))
        if experts and i == case["layers"] - 1 and i > 0:
            mx["kv_from"] = i - 1
        mlp = dict(kind="dense", ff=ff)
        if experts and i > 0:
            mlp = dict(kind="moe", expert=dict(ff=eff, limit=7.0), router=dict(experts=experts, top=top), shared=dict(ff=sff, limit=7.0))
        layers.append(dict(type="attention", mixer=mx, mlp=mlp))
    return dict(architecture="Ditilix", width=W, vocab=VOCAB, residual_mult=0.5, logit_scale=1.0, norm=dict(eps=1e-6, groups=4), layers=layers)


def _stack_tensors(case, cj, seed):
    """(name, device tensor).  Mixtures: the embedding carries, per token, the directions of the experts that token's routers choose — a
    trained router decides clearly, and so does this one."""
    g, dt = _gen(seed), _TORCH[case["dtype"]]
    W = cj["width"]
    experts = STACK[case["model"]][5]
    embed = torch.randn((VOCAB, W), generator=g, device="cuda")
    dirs = None
    if experts:
        dirs = torch.linalg.qr(torch.randn((W, experts), generator=g, device="cuda"))[0].T * math.sqrt(W)
        pick = torch.rand((VOCAB, experts), generator=g, device="cuda").topk(cj["layers"][1]["mlp"]["router"]["top"], dim=1).indices
        embed = embed + 0.5 * dirs[pick].sum(1)
    yield "embed", embed.to(dt)
    yield "head", _normal(g, (VOCAB, W), W ** -0.5, dt)
    yield "final.norm", _normal(g, (W,), 0.1, dt, 1.0)
    for i, layer in enumerate(cj["layers"]):
        p, mx, ml = "l%d." % i, layer["mixer"], layer["mlp"]
        nq, nk, nv = mx["heads"] * mx["dim"], mx["kv_heads"] * mx["dim"], mx["kv_heads"] * mx["vdim"]
        yield p + "norm1", _normal(g, (W,), 0.02, dt, 1.0)
        yield p + "mix.q", _normal(g, (nq, W), W ** -0.5, dt)
        if mx.get("kv_from") is None:
            yield p + "mix.k", _normal(g, (nk, W), W ** -0.5, dt)
            yield p + "mix.v", _normal(g, (nv, W), W ** -0.5, dt)
        yield p + "mix.o", _normal(g, (W, nq), 0.5 * nq ** -0.5, dt)
        if ml["kind"] == "dense":
            yield p + "mlp.up", _normal(g, (ml["ff"], W), W ** -0.5, dt)
            yield p + "mlp.down", _normal(g, (W, ml["ff"]), 0.5 * ml["ff"] ** -0.5, dt)
            yield p + "mlp.act", torch.tensor([0.6, 0.3, 0.1, 0.02], device="cuda").to(dt)
            continue
        yield p + "mlp.router", ((dirs / W) * 6.0 + torch.randn((experts, W), generator=g, device="cuda") * (0.2 * W ** -0.5)).to(dt)
        for e in [("e%d." % e, ml["expert"]["ff"]) for e in range(experts)] + [("shared.", ml["shared"]["ff"])]:
            q, f = p + "mlp." + e[0], e[1]
            yield q + "gate", _normal(g, (f, W), W ** -0.5, dt)
            yield q + "up", _normal(g, (f, W), W ** -0.5, dt)
            yield q + "down", _normal(g, (W, f), 0.3 * f ** -0.5, dt)
        yield p + "mlp.shared.sg", _normal(g, (1, W), W ** -0.5, dt)


def _token_ids(case, seed):
    r = np.random.default_rng(1000003 * int(seed) + 17)
    extra = 1 if case["phase"] == "decode" else 0
    return [r.integers(0, VOCAB, n + extra).astype(np.uint32) for n in _lens(case)]


def _pages(lens, seed):
    """block tables of the sequences over one shuffled pool"""
    need = [(n + BS - 1) // BS for n in lens]
    order = np.random.default_rng(31 * int(seed) + 5).permutation(sum(need)).astype(np.uint32)
    tables, at = np.zeros((len(lens), max(need)), np.uint32), 0
    for i, n in enumerate(need):
        tables[i, :n] = order[at:at + n]
        at += n
    return tables, sum(need)


def _step(ids, starts, tables, decode):
    """arguments of forward_raw for tokens ids[i] at positions starts[i].. of every sequence"""
    pos = np.concatenate([np.arange(s, s + len(t)) for t, s in zip(ids, starts)]).astype(np.int64)
    slots = np.concatenate([tables[i, np.arange(s, s + len(t)) // BS].astype(np.int64) * BS + np.arange(s, s + len(t)) % BS
                            for i, (t, s) in enumerate(zip(ids, starts))])
    ctx = np.array([s + len(t) for t, s in zip(ids, starts)], np.uint32)
    cu = None if decode else np.concatenate([[0], np.cumsum([len(t) for t in ids])]).astype(np.uint32)
    return np.concatenate(ids), pos, slots, tables, ctx, cu


def _prepare_model(case, seed):
    ids = _token_ids(case, seed)
    lens = [len(t) for t in ids]
    tables, blocks = _pages(lens, seed)
    kw = dict(num_gpu_blocks=blocks + 1, max_num_seqs=len(ids), max_model_len=max(lens) + BS, use_graph=False)
    if case["kind"] == "llama":
        cfg = _llama_cfg(case)
        eng = eng_mod.Engine(cfg, fp8_kvcache=case["fp8"], **kw)
        tensors = _llama_tensors(case, cfg, seed)
    else:
        from vllm_rs_amd import checkpoint
        cj = _stack_json(case)
        eng = eng_mod.Engine(checkpoint.parse_config(cj, "float32" if case["dtype"] == "f32" else None), **kw)
        tensors = _stack_tensors(case, cj, seed)
    for name, t in tensors:
        eng.load_weights({name: _host(t)}, finalize=False)
    eng.finalize()
    if case["phase"] == "prompt":
        return dict(kind="model", eng=eng, args=_step(ids, [0] * len(ids), tables, False))
    for i, t in enumerate(ids):  # the contexts' cache rows
        for at in range(0, len(t) - 1, 8192):
            part = t[at:min(at + 8192, len(t) - 1)]
            eng.forward_raw(*_step([part], [at], tables[i:i + 1], False))
    return dict(kind="model", eng=eng, args=_step([t[-1:] for t in ids], [len(t) - 1 for t in ids], tables, True))


def _scan_inputs(case, seed):
    g, H, D = _gen(seed), case["heads"], case["dim"]
    G, T = H // case["rep"], sum(_lens(case))
    unit = lambda t: t / t.norm(dim=-1, keepdim=True)
    return dict(q=unit(torch.randn((T, G, D), generator=g, device="cuda")), k=unit(torch.randn((T, G, D), generator=g, device="cuda")),
                v=torch.randn((T, H, D), generator=g, device="cuda"), decay=torch.rand((T, H, D), generator=g, device="cuda") * 0.1 + 0.9,
                beta=torch.rand((T, H), generator=g, device="cuda"))


def _latent_inputs(case, seed):
    g, H, kd, lens = _gen(seed), case["heads"], case["rank"] + case["rot"], _lens(case)
    tables, blocks = _pages(lens, seed)
    rows = _normal(g, (blocks * BS, kd), 1.0, torch.bfloat16)
    return dict(q=_normal(g, (len(lens), H, kd), 1.5, torch.bfloat16), rows=rows, tables=tables, gate=torch.randn((len(lens), H), generator=g, device="cuda"))


def prepare(case, seed):
    if case["kind"] in ("llama", "stack"):
        return _prepare_model(case, seed)
    lens = _lens(case)
    dev = lambda a, t: torch.tensor(np.asarray(a).astype(t), device="cuda")
    if case["kind"] == "scan":
        s, H, D = _scan_inputs(case, seed), case["heads"], case["dim"]
        s.update(kind="scan", case=dict(case), state=torch.zeros((len(lens), H, D, D), device="cuda"), out=torch.empty_like(s["v"]),
                 slots=dev(range(len(lens)), np.int32), positions=dev(np.concatenate([np.arange(n) for n in lens]), np.int64),
                 cu=dev(np.concatenate([[0], np.cumsum(lens)]), np.int32))
        return s
    s = _latent_inputs(case, seed)
    B, H = len(lens), case["heads"]
    splits = min(32, (max(lens) + 63) // 64)
    s.update(kind="latent", case=dict(case), dtables=dev(s["tables"].view(np.int32), np.int32), ctx=dev(lens, np.int32), splits=splits,
             positions=dev(np.array(lens) - 1, np.int64), out=torch.empty((B, H, case["rank"]), device="cuda", dtype=torch.bfloat16),
             scratch=torch.empty(B * splits * H * (case["rank"] + 2), device="cuda"))
    return s


# ---------------------------------------------------------------------------------------------------------------- one pass
def run(state):
    if state["kind"] == "model":
        return state["eng"].forward_raw(*state["args"])
    L, s, case = _lib.load(), state, state["case"]
    stream = torch.cuda.current_stream().cuda_stream
    H = case["heads"]
    if s["kind"] == "scan":
        G, D = H // case["rep"], case["dim"]
        L.vra_stack_op_linear_scan(s["q"].data_ptr(), G * D, s["k"].data_ptr(), G * D, s["v"].data_ptr(), H * D, s["decay"].data_ptr(), H * D, None,
                                   s["beta"].data_ptr(), H, D ** -0.5, s["state"].data_ptr(), s["slots"].data_ptr(), s["positions"].data_ptr(),
                                   s["cu"].data_ptr(), s["out"].data_ptr(), H * D, case["seqs"], H, case["rep"], D, D, stream)
        return dict(out=s["out"], state=s["state"])
    kd, rank = case["rank"] + case["rot"], case["rank"]
    B = case["seqs"]
    L.vra_stack_op_attention_latent(s["q"].data_ptr(), H * kd, s["out"].data_ptr(), s["rows"].data_ptr(), kd, s["positions"].data_ptr(), s["dtables"].data_ptr(),
                                    s["ctx"].data_ptr(), None, B, B, 1, H, kd, rank, BS, s["dtables"].shape[1], (128 + case["rot"]) ** -0.5, 0, None, None,
                                    s["gate"].data_ptr(), H, s["scratch"].data_ptr(), s["scratch"].numel() * 4, s["splits"], 0, stream)
    return dict(out=s["out"])


# ---------------------------------------------------------------------------------------------------------------- what a pass needs
def work(case):
    lens = _lens(case)
    if case["kind"] == "scan":
        T, H, D = sum(lens), case["heads"], case["dim"]
        return dict(bytes=4 * (T * (2 * (H // case["rep"]) * D + 3 * H * D + H) + len(lens) * H * D * D), flops=T * H * D * D * 7)
    if case["kind"] == "latent":
        H, kd, rank = case["heads"], case["rank"] + case["rot"], case["rank"]
        return dict(bytes=sum(lens) * kd * 2 + len(lens) * H * (kd + rank) * 2, flops=sum(lens) * H * 2 * (kd + rank))
    decode = case["phase"] == "decode"
    T = len(lens) if decode else sum(lens)
    pairs = sum(lens) + len(lens) if decode else sum(n * (n + 1) // 2 for n in lens)  # (query, key) pairs of one head
    seen = sum(lens) + len(lens) if decode else 0  # cache rows read that this step does not write
    es = 4 if case["dtype"] == "f32" else 2
    if case["kind"] == "llama":
        cfg = _llama_cfg(case)
        n = sum(K * N for K, N in _llama_shapes(cfg).values())
        wb = n * 2 if case["quant"] == "none" else n // 2 + n // cfg["group_size"] * (2 if case["quant"] == "gptq" else 2.5)
        H, D, kvd = cfg["hidden_size"], cfg["head_dim"], cfg["num_kv_heads"] * cfg["head_dim"]
        layer_b = wb + (seen + T) * 2 * kvd * (1 if case["fp8"] else 2)
        layer_f = 2 * n * T + 4 * pairs * cfg["num_heads"] * D
        b, f = cfg["num_layers"] * layer_b, cfg["num_layers"] * layer_f
    else:
        cj = _stack_json(case)
        H, b, f = cj["width"], 0, 0
        for layer in cj["layers"]:
            mx, ml = layer["mixer"], layer["mlp"]
            own = mx.get("kv_from") is None
            n = H * mx["heads"] * (mx["dim"] + mx["vdim"]) + (H * mx["kv_heads"] * (mx["dim"] + mx["vdim"]) if own else 0)
            used = n
            if ml["kind"] == "dense":
                n, used = n + 2 * H * ml["ff"], used + 2 * H * ml["ff"]
            else:
                one, ro = 3 * H * ml["expert"]["ff"], ml["router"]
                n += min(ro["experts"], T * ro["top"]) * one + 3 * H * ml["shared"]["ff"] + H * ro["experts"]
                used += ro["top"] * one + 3 * H * ml["shared"]["ff"] + H * ro["experts"]
            b += n * es + (seen + T) * mx["kv_heads"] * (mx["dim"] + mx["vdim"]) * es
            f += 2 * used * T + 2 * pairs * mx["heads"] * (mx["dim"] + mx["vdim"])
    rows = len(lens)
    return dict(bytes=b + VOCAB * H * es + T * H * es + rows * VOCAB * 4, flops=f + 2 * rows * VOCAB * H)


def tolerance(case):
    """four times the distance from the 64-bit result that was measured: bf16 rounds eight times as coarsely as f16, the small decoder's
    six narrow layers amplify more than the wide ones', the FP8 cache's rounding dominates whatever the 16-bit type"""
    if case["kind"] == "scan":
        return dict(rel=2e-6)
    if case["kind"] == "latent":
        return dict(rel=8e-3)
    if case["dtype"] == "f32":
        return dict(rel=2e-5)
    if case["kind"] == "stack":
        return dict(rel=8e-3)
    if case["dtype"] == "f16" and not case["fp8"]:
        return dict(rel=5e-3 if case["model"] == "tinyllama" else 2.5e-3)
    return dict(rel=0.03 if case["model"] == "tinyllama" else 0.018)


# ---------------------------------------------------------------------------------------------------------------- in 64 bits
def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _attend(q, k, v, scale, softcap=0.0):
    """causal softmax attention of one sequence's last rows: q [Tq, H, D] over k, v [T, G, .]"""
    Tq, H, T, G = q.shape[0], q.shape[1], k.shape[0], k.shape[1]
    out = torch.empty((Tq, H, v.shape[2]), dtype=torch.float64, device="cuda")
    at = torch.arange(T, device="cuda")
    for h in range(H):
        kh, vh = k[:, h * G // H].contiguous(), v[:, h * G // H].contiguous()
        for a in range(0, Tq, 4096):
            s = (q[a:a + 4096, h] @ kh.T) * scale
            if softcap:
                s = softcap * torch.tanh(s / softcap)
            s = s.masked_fill(at[None, :] > at[T - Tq + a:T - Tq + a + s.shape[0], None], float("-inf"))
            out[a:a + 4096, h] = torch.softmax(s, -1) @ vh
    return out


def _unpack(t, case, cfg, w, p):
    """the [K, N] weight of an int4 (or dense) projection"""
    if case["quant"] == "none":
        return w[p + ".weight"].double().T
    codes, zeros, s = w[p + ".qweight"], w[p + ".qzeros"], w[p + ".scales"].double()
    if case["quant"] == "gptq":  # eight rows a word
        q = torch.stack([(codes >> (4 * i)) & 15 for i in range(8)], 1).reshape(codes.shape[0] * 8, codes.shape[1])
        z = torch.full_like(s, 8.0)
    else:  # eight columns a word, in the order 0 2 4 6 1 3 5 7
        shifts = [0, 4, 1, 5, 2, 6, 3, 7]
        q = torch.stack([(codes >> (4 * i)) & 15 for i in shifts], 2).reshape(codes.shape[0], -1)
        z = torch.stack([(zeros >> (4 * i)) & 15 for i in shifts], 2).reshape(zeros.shape[0], -1).double()
    g = cfg["group_size"]
    K, N = q.shape
    return ((q.double().reshape(K // g, g, N) - z[:, None]) * s[:, None]).reshape(K, N)


def _rotate(x, theta):
    T, _, D = x.shape
    ang = torch.arange(T, device="cuda", dtype=torch.float64)[:, None] * theta ** (-torch.arange(0, D, 2, device="cuda", dtype=torch.float64) / D)
    c, s = ang.cos()[:, None], ang.sin()[:, None]
    a, b = x[..., :D // 2], x[..., D // 2:]
    return torch.cat([a * c - b * s, b * c + a * s], -1)


def _exact_llama(case, seed):
    cfg = _llama_cfg(case)
    w = dict(_llama_tensors(case, cfg, seed))
    D, eps = cfg["head_dim"], cfg["rms_norm_eps"]
    ids = _token_ids(case, seed)
    cut = np.cumsum([0] + [len(t) for t in ids])
    x = w["model.embed_tokens.weight"][torch.tensor(np.concatenate(ids).astype(np.int64), device="cuda")].double()
    for i in range(cfg["num_layers"]):
        p = "model.layers.%d." % i
        lin = lambda h, n: h @ _unpack(None, case, cfg, w, p + n) + (w[p + n + ".bias"].double() if p + n + ".bias" in w else 0.0)
        h = _rms(x, eps) * w[p + "input_layernorm.weight"].double()
        q, k, v = (lin(h, "self_attn.%s_proj" % n).reshape(len(x), -1, D) for n in "qkv")
        o = torch.empty_like(q)
        for a, b in zip(cut, cut[1:]):
            qs, ks, vs = _rotate(q[a:b], cfg["rope_theta"]), _rotate(k[a:b], cfg["rope_theta"]), v[a:b]
            if case["fp8"]:  # the cache's element type is part of the model's definition
                ks, vs = (t.float().clamp(-448, 448).to(torch.float8_e4m3fn).double() for t in (ks, vs))
            o[a:b] = _attend(qs, ks, vs, D ** -0.5)
        x = x + lin(o.reshape(len(x), -1), "self_attn.o_proj")
        h = _rms(x, eps) * w[p + "post_attention_layernorm.weight"].double()
        act = torch.nn.functional.silu(lin(h, "mlp.gate_proj")) * lin(h, "mlp.up_proj")
        x = x + lin(act, "mlp.down_proj")
    last = torch.tensor(cut[1:] - 1, device="cuda")
    return (_rms(x[last], eps) * w["model.norm.weight"].double()) @ w["lm_head.weight"].double().T


def _exact_stack(case, seed):
    cj = _stack_json(case)
    w = dict(_stack_tensors(case, cj, seed))
    W, eps, groups = cj["width"], cj["norm"]["eps"], cj["norm"]["groups"]
    d = lambda n: w[n].double()
    norm = lambda x, n: _rms(x.reshape(len(x), groups, -1), eps).reshape(len(x), W) * d(n)
    expert = lambda h, p: _glu(h @ d(p + "gate").T, h @ d(p + "up").T) @ d(p + "down").T
    ids = _token_ids(case, seed)
    cut = np.cumsum([0] + [len(t) for t in ids])
    pos = torch.tensor(np.concatenate([np.arange(len(t)) for t in ids]), device="cuda").double()
    x = w["embed"][torch.tensor(np.concatenate(ids).astype(np.int64), device="cuda")].double()
    ang = pos[:, None] * 10000.0 ** (-2.0 * torch.arange(W // 2, device="cuda", dtype=torch.float64) / W)
    x = x + torch.stack([ang.sin(), ang.cos()], -1).reshape(len(x), W)
    kv = {}
    for i, layer in enumerate(cj["layers"]):
        p, mx, ml = "l%d." % i, layer["mixer"], layer["mlp"]
        h = norm(x, p + "norm1")
        src = mx.get("kv_from", i)
        q = (h @ d(p + "mix.q").T).reshape(len(x), mx["heads"], -1)
        q = q * (1.0 + mx["q_temp"]["coef"] * torch.log(torch.floor((pos + 1) / mx["q_temp"]["every"]) + 1.0))[:, None, None]
        if src == i:
            kv[i] = [(h @ d(p + "mix." + n).T).reshape(len(x), mx["kv_heads"], -1) for n in "kv"]
        o = torch.cat([_attend(q[a:b], kv[src][0][a:b], kv[src][1][a:b], mx["scale"], mx["softcap"]) for a, b in zip(cut, cut[1:])])
        o = o.reshape(len(x), -1) @ d(p + "mix.o").T
        if ml["kind"] == "dense":
            z = h @ d(p + "mlp.up").T
            c = d(p + "mlp.act")
            ff = (c[0] * _rms(z, eps) + c[1] * _rms(z * z, eps) + c[2] * _rms(z * z * z, eps) + c[3]) @ d(p + "mlp.down").T
        else:
            ff = torch.sigmoid(h @ d(p + "mlp.shared.sg").T) * expert(h, p + "mlp.shared.")
            score, pick = torch.sigmoid(h @ d(p + "mlp.router").T).topk(ml["router"]["top"], dim=1)
            for e in range(ml["router"]["experts"]):
                t, j = torch.nonzero(pick == e, as_tuple=True)
                if len(t):
                    ff[t] += expert(score[t, j, None] * h[t], p + "mlp.e%d." % e)
        x = x + cj["residual_mult"] * (o + ff)
    last = torch.tensor(cut[1:] - 1, device="cuda")
    return norm(x[last], "final.norm") @ d("head").T


def _glu(g, u, limit=7.0):
    g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return g * torch.sigmoid(1.702 * g) * (u + 1.0)


def exact(case, seed):
    if case["kind"] == "llama":
        return _exact_llama(case, seed).cpu().numpy()
    if case["kind"] == "stack":
        return _exact_stack(case, seed).cpu().numpy()
    lens = _lens(case)
    if case["kind"] == "scan":
        s, D = {k: t.double() for k, t in _scan_inputs(case, seed).items()}, case["dim"]
        q, k = (s[n].repeat_interleave(case["rep"], 1) for n in "qk")
        out, states, at = torch.empty_like(s["v"]), [], 0
        for n in lens:
            S = torch.zeros((case["heads"], D, D), dtype=torch.float64, device="cuda")  # [value, key]
            for t in range(at, at + n):
                S = S * s["decay"][t][:, None, :]
                u = s["beta"][t][:, None] * (s["v"][t] - (S * k[t][:, None, :]).sum(-1))
                S = S + u[:, :, None] * k[t][:, None, :]
                out[t] = (S * q[t][:, None, :]).sum(-1) * D ** -0.5
            states.append(S)
            at += n
        return dict(out=out, state=torch.stack(states))
    s, rank = _latent_inputs(case, seed), case["rank"]
    out = []
    for i, n in enumerate(lens):
        slot = s["tables"][i, np.arange(n) // BS].astype(np.int64) * BS + np.arange(n) % BS
        rows = s["rows"][torch.tensor(slot, device="cuda")].double()
        a = torch.softmax((s["q"][i].double() @ rows.T) * (128 + case["rot"]) ** -0.5, -1) @ rows[:, :rank]
        out.append(a * torch.sigmoid(s["gate"][i].double())[:, None])
    return dict(out=torch.stack(out))
