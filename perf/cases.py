"""The work that a user of the engine has it do, as cases that can be timed and compared.

A case is a dict of plain values; ``kind`` says which calls it makes:

  decode    one sequence of a GGUF model, some tokens one after the other from a given context (`HipGpuInference.forward`: logits to the host
            after every token, what a sampler reads)
  prompt    one sequence's prompt from nothing, logits after its last token (`eval`)
  batch     several sequences: their prompts, then some tokens each, all sequences a step (`batch_reset`, `batch_prefill`, `forward_multi`)
  generate  a model described layer by layer: a prompt from nothing, then some tokens one after the other (`reset`, `eval`, `forward`)

Widths, heads, vocabularies and quantisations are those of the package's configurations and of the benchmark's layer-by-layer sizes; most cases keep
the real widths and take some of the layers (a layer is a layer: the others repeat it).  Weights are random blocks of the real formats,
tokens are random.  ``exact`` is the same model in 64 bits, written here from the formats and formulas alone.
"""
from __future__ import annotations

import importlib
import math

import numpy as np
import torch

lg = importlib.import_module("llama-gguf_amd")

KV_TYPES = {"f32": 0, "tq2": 4, "tq3": 5}

# ---- the cases -------------------------------------------------------------------------------------------------------------------


def listed():
    return [
        # a small model answering in a chat: every call is short, launches and their gaps count
        dict(name="decode-small", kind="decode", model="tinyllama-1.1b", mix="Q4_K_M", layers=22, vocab=32000, context=40, steps=4, kv="f32"),
        # the benchmark's own workload: the whole 8B model, one sequence, behind a short prompt
        dict(name="decode-8b", kind="decode", model="llama-3-8b", mix="Q4_K_M", layers=32, vocab=128256, context=128, steps=8, kv="f32"),
        # a long conversation with a model of the widest format: the cache counts beside the weights
        dict(name="decode-long", kind="decode", model="llama-3-8b", mix="Q8_0", layers=8, vocab=32000, context=3001, steps=8, kv="f32"),
        # the compressed cache that the command line offers, on the middle quantisation
        dict(name="decode-tq3", kind="decode", model="llama-3-8b", mix="Q5_K_M", layers=8, vocab=32000, context=500, steps=8, kv="tq3"),
        # a mixture of experts, one sequence: two of eight experts a token
        dict(name="decode-moe", kind="decode", model="mixtral-8x7b", mix="Q5_K_M", layers=3, vocab=32000, context=200, steps=8, kv="f32"),
        # a server's step with all its slots taken, prompts of different lengths
        dict(name="batch-16", kind="batch", model="llama-3-8b", mix="Q4_K_M", layers=8, vocab=32000, sequences=16, shortest=11, longest=100, steps=24, kv="f32"),
        # a server with a few sequences on a mixture of experts, from their opening tokens on
        dict(name="batch-moe-5", kind="batch", model="mixtral-8x7b", mix="Q5_K_M", layers=2, vocab=32000, sequences=5, shortest=0, longest=0, steps=24, kv="f32"),
        # the benchmark's prompt, an ordinary question
        dict(name="prompt-128", kind="prompt", model="llama-3-8b", mix="Q4_K_M", layers=32, vocab=128256, tokens=128),
        # a document in the prompt, an odd number of tokens
        dict(name="prompt-2047", kind="prompt", model="llama-3-8b", mix="Q4_K_M", layers=16, vocab=32000, tokens=2047),
        # a page of text for a mixture of experts
        dict(name="prompt-moe-600", kind="prompt", model="mixtral-8x7b", mix="Q5_K_M", layers=2, vocab=32000, tokens=600),
        # a document for a model described layer by layer (attention with windows and shared keys, delta rule, query latents), then an answer's start
        dict(name="layers-prompt", kind="generate", design="Tarudra", width=2048, ff=5632, vocab=32000, layers=8, heads=16, prompt=1501, steps=2),
        # an answer of a model described layer by layer (latent attention and matrix memory), after a short prompt
        dict(name="layers-answer", kind="generate", design="Zamelix", width=4096, ff=14336, vocab=32000, layers=4, heads=32, prompt=77, steps=24),
    ]


def _spread(rng, lo, hi):
    """A whole number between lo and hi, even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(("decode", "decode", "prompt", "prompt", "batch", "generate"))
    if kind == "generate":
        design = rng.choice(("Tarudra", "Zamelix"))
        width = rng.choice((2048, 2048, 4096))
        return dict(kind=kind, design=design, width=width, ff={2048: 5632, 4096: 14336}[width], vocab=32000, layers=4 if width == 4096 else rng.choice((4, 8)),
                    heads=width // 128, prompt=_spread(rng, 17, 1500), steps=rng.randint(2, 16))
    model = rng.choice(("tinyllama-1.1b", "llama-3-8b", "llama-3-8b", "mixtral-8x7b"))
    mix = "Q5_K_M" if model == "mixtral-8x7b" else rng.choice(("Q4_K_M", "Q4_K_M", "Q5_K_M", "Q8_0", "Q4_0"))
    layers = {"tinyllama-1.1b": rng.randint(4, 22), "llama-3-8b": rng.randint(2, 8), "mixtral-8x7b": rng.randint(1, 2)}[model]
    case = dict(kind=kind, model=model, mix=mix, layers=layers, vocab=32000)
    if kind == "decode":
        kv = rng.choice(("f32", "f32", "f32", "tq3", "tq2"))
        return dict(case, context=_spread(rng, 1, 3000 if kv == "f32" and model != "mixtral-8x7b" else 600), steps=rng.randint(2, 8), kv=kv)
    if kind == "prompt":
        return dict(case, tokens=_spread(rng, 9, 2047))
    # (prompt blocks round operands to 16 bits, after which a router's close call may fall to either side: mixtures start with steps)
    longest = 0 if model == "mixtral-8x7b" else _spread(rng, 12, 100)
    return dict(case, sequences=rng.randint(2, 16), shortest=rng.randint(min(2, longest), longest), longest=longest, steps=rng.randint(8, 24), kv="f32")


# ---- inputs ----------------------------------------------------------------------------------------------------------------------


def _gguf_model(case, seed):
    cfg = lg.make_config(case["model"], max_seq_len=_room(case), num_layers=case["layers"], vocab_size=case["vocab"])
    return lg.SynthModel(cfg, mix=case["mix"], seed=(0x9E3779B97F4A7C15 * (seed + 1)) & 0xFFFFFFFFFFFFFFFF)


def _room(case):
    """Positions that the context is made for."""
    if case["kind"] == "decode":
        return case["context"] + case["steps"] + 8
    if case["kind"] == "batch":
        return case["longest"] + case["steps"] + 8
    return case["tokens"] + 8 if case["kind"] == "prompt" else case["prompt"] + case["steps"] + 8


def _ids(case, seed, n, which=0):
    return np.random.default_rng([seed, which, 7]).integers(0, case["vocab"], n).astype(np.uint32)


def _lengths(case, seed):
    """Prompt lengths of the sequences of a batch."""
    a, b, n = case["shortest"], case["longest"], case["sequences"]
    return [int(v) for v in np.random.default_rng([seed, 3]).permutation(np.linspace(a, b, n).round())]


def _signs(case, cfg, seed):
    """The rotations' signs of the compressed caches, [layer][kv head][key, value][head size]."""
    if case.get("kv", "f32") == "f32":
        return None
    return np.random.default_rng([seed, 5]).choice(np.array([-1.0, 1.0], np.float32), (cfg.num_layers, cfg.num_kv_heads, 2, cfg.head_dim))


class _Layered:
    """Weights of a model described layer by layer, made by name from the seed on the GPU: bf16, scaled by 1 / sqrt(in)."""

    def __init__(self, seed):
        self.seed = seed

    def tensor(self, name, shape):
        g = torch.Generator(device="cuda")
        h = self.seed + 1
        for ch in name:
            h = (h * 1000003 + ord(ch)) & 0x7FFFFFFF
        g.manual_seed(h)
        v = torch.randn(shape, generator=g, device="cuda", dtype=torch.float32)
        last = name.split(".")[-1]
        if last in ("ls1", "ls2"):
            v = 0.7 + 0.2 * v
        elif last == "dt_bias":
            v = -4.0 + 1.5 * v              # a state that lasts
        elif name.endswith(".f.b"):
            v = 3.0 + v                     # a memory that lasts
        elif last == "conv":
            v = 0.5 * v
        elif "norm" in last:
            v = 1.0 + 0.2 * v
        elif len(shape) == 1:
            v = 0.5 * v
        elif name not in ("embed", "bigram"):
            v = v / math.sqrt(shape[1])
        return v.to(torch.bfloat16)

    def get(self, name, shape):
        return 30, self.tensor(name, shape).view(torch.int16).cpu().numpy().view(np.uint16).reshape(-1)


def _layered_config(case):
    W, H = case["width"], case["heads"]
    if case["design"] == "Tarudra":
        mlp, mask = {"kind": "dense", "ff": case["ff"]}, {"size": 1024 if W == 2048 else 8192}
        grouped = {"heads": H, "kv_heads": H // 4, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "mask": mask,
                   "rot": {"base": 10000.0, "dims": 128, "scaling": {"factor": 4.0, "original": 4096, "fast": 32.0, "slow": 1.0}}}
        delta = {"heads": H, "kv_heads": H // 2, "dim": 128, "vdim": 128, "conv": 4}
        latent = {"heads": H, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "q_rank": 768 * W // 2048, "scale": 192 ** -0.5, "mask": mask,
                  "rot": {"base": 10000.0, "dims": 64}}
        turn = [("attention", lambda i: grouped), ("delta", lambda i: delta), ("attention", lambda i: dict(grouped, kv_from=i - 2)),
                ("latent_attention", lambda i: latent)]
        return {"architecture": "Tarudra", "width": W, "vocab": case["vocab"], "norm": {"eps": 1e-5}, "logit_softcap": 30.0,
                "layers": [{"type": turn[i % 4][0], "mixer": turn[i % 4][1](i), "mlp": mlp} for i in range(case["layers"])]}
    attn = {"type": "latent_attention", "mlp": {"kind": "dense", "ff": case["ff"]},
            "mixer": {"heads": H, "dim": 128, "rot_dim": 64, "vdim": 128, "kv_rank": 512, "scale": 192 ** -0.5, "rot": {"base": 10000.0, "dims": 64}}}
    mem = {"type": "mlstm", "mlp": None, "mixer": {"heads": H // 4, "dim": 256, "vdim": 512, "gate_cap": 15.0}}
    return {"architecture": "Zamelix", "width": W, "vocab": case["vocab"], "norm": {"eps": 1e-5}, "residual_mult": 0.5,
            "embedding": {"bigram": {"buckets": 4096, "mul_prev": 31, "mul_cur": 7}}, "layers": [mem if i % 2 else attn for i in range(case["layers"])]}


def prepare(case, seed):
    if case["kind"] == "generate":
        parsed = lg.layered_model.parse_config(_layered_config(case))
        gpu = lg.HipGpuInference.from_layered(lg.LayeredModel(parsed, _Layered(seed)), _room(case))
        return dict(case=case, gpu=gpu, prompt=_ids(case, seed, case["prompt"]), after=[int(t) for t in _ids(case, seed, case["steps"], 1)])
    model = _gguf_model(case, seed)
    gpu = lg.HipGpuInference.from_model(model, _room(case), kv_cache_type=KV_TYPES[case.get("kv", "f32")], kv_rotation_signs=_signs(case, model.config, seed))
    if case["kind"] == "prompt":
        return dict(case=case, gpu=gpu, prompt=_ids(case, seed, case["tokens"]))
    if case["kind"] == "decode":
        before = _ids(case, seed, case["context"])
        if case["context"] > 600:
            gpu.forward_batch(before)
        else:                                # as GpuModelWrapper feeds a prompt
            for t in before:
                gpu.prefill_token(int(t))
        gpu.synchronize()
        return dict(case=case, gpu=gpu, after=[int(t) for t in _ids(case, seed, case["steps"], 1)])
    gpu.batch_create(case["sequences"])
    prompts = [_ids(case, seed, n, 10 + s) for s, n in enumerate(_lengths(case, seed))]
    return dict(case=case, gpu=gpu, prompts=prompts, slots=list(range(case["sequences"])),
                after=_ids(case, seed, case["steps"] * case["sequences"], 1).reshape(case["steps"], case["sequences"]))


def run(state):
    case, gpu = state["case"], state["gpu"]
    if case["kind"] == "decode":
        gpu.kv_truncate(case["context"])
        return [gpu.forward(t) for t in state["after"]]
    if case["kind"] == "prompt":
        gpu.reset()
        return gpu.eval(state["prompt"], [case["tokens"] - 1])
    if case["kind"] == "generate":
        gpu.reset()
        return [gpu.eval(state["prompt"], [case["prompt"] - 1])] + [gpu.forward(t) for t in state["after"]]
    for s in state["slots"]:
        gpu.batch_reset(s)
        if len(state["prompts"][s]):
            gpu.batch_prefill(s, state["prompts"][s])
    return [gpu.forward_multi(state["slots"], toks)[0] for toks in state["after"]]


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------------

BYTES_PER_WEIGHT = {"Q4_K": 144 / 256, "Q5_K": 176 / 256, "Q6_K": 210 / 256, "Q8_0": 34 / 32, "Q4_0": 18 / 32}
CACHE_BYTES = {"f32": 4.0, "tq2": 0.25, "tq3": 0.375}     # per cached value


def _gguf_work(case):
    cfg = lg.make_config(case["model"], num_layers=case["layers"], vocab_size=case["vocab"])
    base = case["mix"][:-2] if case["mix"].endswith("_M") else case["mix"]
    b = BYTES_PER_WEIGHT[base]
    W, kvw, qw, V, L = cfg.hidden_size, cfg.num_kv_heads * cfg.head_dim, cfg.num_heads * cfg.head_dim, cfg.vocab_size, cfg.num_layers
    ff, E, top = cfg.expert_intermediate_size or cfg.intermediate_size, max(1, cfg.num_experts), max(1, cfg.num_experts_per_token)
    attn_w, expert_w = W * (2 * qw + 2 * kvw), 3 * W * ff
    heads_b = BYTES_PER_WEIGHT["Q6_K"] if case["mix"].endswith("_M") else b
    row = 2 * kvw * CACHE_BYTES[case.get("kv", "f32")] * L                    # cache bytes of a position

    def weights(experts):                                                      # bytes of all matrices of the layers; the _M mixes hold a part of v and down wider
        wide = 0.5 * (heads_b - b) * (W * kvw + W * ff * experts) if case["mix"].endswith("_M") else 0.0
        return L * (b * (attn_w + expert_w * experts) + wide)

    def flops(tokens, seen, logits):
        return tokens * 2 * L * (attn_w + expert_w * top) + 4 * L * qw * seen + logits * 2 * W * V
    some = lambda n: E * (1 - (1 - top / E) ** n)                              # experts that n tokens choose between them
    if case["kind"] == "decode":
        n, seen = case["steps"], sum(case["context"] + i + 1 for i in range(case["steps"]))
        return n * (weights(top) + heads_b * W * V + 4 * V) + row * (seen + n), flops(n, seen, n)
    if case["kind"] == "prompt":
        n = case["tokens"]
        return weights(some(n)) + heads_b * W * V + 4 * V + 2 * row * n, flops(n, n * (n + 1) / 2, 1)
    B, n, mean = case["sequences"], case["steps"], (case["shortest"] + case["longest"]) / 2
    p, seen = B * mean, B * sum(mean + i + 1 for i in range(case["steps"]))
    prompts = (B * weights(some(mean)) if mean else 0) + 2 * row * p           # one prompt a call
    return prompts + n * (weights(some(B)) + heads_b * W * V + B * 4 * V) + row * (seen + B * n), flops(p, B * mean * mean / 2, 0) + flops(B * n, seen, B * n)


def _layered_work(case):
    W, H, V, n, s = case["width"], case["heads"], case["vocab"], case["prompt"], case["steps"]
    cfg = _layered_config(case)
    parsed = lg.layered_model.parse_config(cfg)
    mats = sum(math.prod(sh) for name, sh in parsed.tensor_shapes() if name not in ("embed", "bigram", "head"))
    flops, cache = (n + s) * 2.0 * mats + (1 + s) * 2.0 * W * V, 0.0
    for lay in cfg["layers"]:
        mx = lay["mixer"]
        if "attention" in lay["type"]:
            seen = sum(min(i + 1, mx.get("mask", {"size": 1 << 30})["size"]) for i in range(n + s))
            flops += 2.0 * H * seen * (mx["dim"] + mx.get("rot_dim", 0) + mx["vdim"])
            row = 2 * (mx["kv_rank"] + mx["rot_dim"]) if "kv_rank" in mx else 2 * mx["kv_heads"] * (mx["dim"] + mx["vdim"])
            cache += row * (n + s + s * min(n, mx.get("mask", {"size": 1 << 30})["size"]))
        else:
            flops += (n + s) * mx["heads"] * 6.0 * mx["dim"] * mx["vdim"]
            cache += 2 * 4 * s * mx["heads"] * mx["dim"] * mx["vdim"]
    return (1 + s) * 2.0 * (mats + W * V) + cache + (1 + s) * 4.0 * V, flops


def work(case):
    b, f = _layered_work(case) if case["kind"] == "generate" else _gguf_work(case)
    return {"bytes": int(b), "flops": int(f)}


def tolerance(case):
    """About four times the largest error against `exact` that was measured: decode steps hold activations in 32 bits (1e-6, mixtures 5e-6); the compressed
    caches pick the other code where a value lies between two (1.4e-4); prompts round the operands of the products to 16 bits, and what follows a
    prompt inherits that (4e-3); bf16 for the layer-by-layer models (7e-3)."""
    if case["kind"] == "generate":
        return {"rel": 2.8e-2, "max": 0.28}
    if case["kind"] == "decode" and case["kv"] != "f32":
        return {"rel": 6e-4, "max": 6e-3}
    if case["kind"] == "decode" and case["context"] <= 600 or case["kind"] == "batch" and case["longest"] == 0:
        return {"rel": 2e-5, "max": 2e-4}
    return {"rel": 1.6e-2, "max": 0.16}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------------------

F64 = torch.float64


def _fields(raw, block, *cuts):
    """Bytes of blocks on the GPU, cut into fields."""
    b, out, at = raw.view(-1, block), [], 0
    for n in cuts:
        out.append(b[:, at:at + n])
        at += n
    return out


def _half(b):
    return b.contiguous().view(torch.float16).to(F64)


def _k_scales(s):
    """The eight 6-bit scales and mins of a K block."""
    s = s.to(torch.int32)
    sc = torch.cat([s[:, 0:4] & 63, (s[:, 8:12] & 15) | ((s[:, 0:4] >> 6) << 4)], 1)
    mn = torch.cat([s[:, 4:8] & 63, (s[:, 8:12] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1)
    return sc.to(F64), mn.to(F64)


def _dequantized(t, raw):
    """A GGUF tensor's values in 64 bits, flat."""
    if t == 0:
        return raw.view(torch.float32).to(F64)
    if t == 8:                                                                  # Q8_0
        d, q = _fields(raw, 34, 2, 32)
        return (_half(d) * q.contiguous().view(torch.int8).to(F64)).reshape(-1)
    if t == 2:                                                                  # Q4_0
        d, q = _fields(raw, 18, 2, 16)
        return (_half(d) * (torch.cat([q & 15, q >> 4], 1).to(F64) - 8.0)).reshape(-1)
    if t == 14:                                                                 # Q6_K
        ql, qh, sc, d = _fields(raw, 210, 128, 64, 16, 2)
        ql, qh = ql.reshape(-1, 2, 2, 32), qh.reshape(-1, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)                                  # [block, half, quarter, 32]
        high = torch.cat([(qh >> (2 * i)) & 3 for i in range(4)], 2)
        q = (low | (high << 4)).to(F64) - 32.0
        s = sc.contiguous().view(torch.int8).to(F64).reshape(-1, 2, 4, 2, 1)
        return (_half(d).view(-1, 1, 1, 1, 1) * s * q.reshape(-1, 2, 4, 2, 16)).reshape(-1)
    five = t == 13                                                              # Q5_K, Q4_K
    parts = _fields(raw, 176 if five else 144, 2, 2, 12, *((32, 128) if five else (128,)))
    d, dmin, (sc, mn), qs = _half(parts[0]), _half(parts[1]), _k_scales(parts[2]), parts[-1].reshape(-1, 4, 1, 32)
    q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32)
    if five:
        q = q | (torch.stack([(parts[3] >> i) & 1 for i in range(8)], 1) << 4)
    return ((d * sc).unsqueeze(2) * q.to(F64) - (dmin * mn).unsqueeze(2)).reshape(-1)


class _Gguf:
    """The model's tensors in 64 bits, one at a time."""

    def __init__(self, model):
        self.model, self.specs = model, {s.name: s for s in model.specs()}

    def matrix(self, name, part=None):
        s = self.specs[name]
        raw = torch.from_numpy(self.model.payload(s)).cuda()
        if part is not None:
            raw = raw.view(s.ne[2], -1)[part].contiguous()
        v = _dequantized(s.ggml_type, raw)
        return v if len(s.ne) == 1 else v.view(-1, s.ne[0])


def _rms(x, eps):
    return x / torch.sqrt(torch.mean(x * x, -1, keepdim=True) + eps)


def _turn_pairs(x, angle):
    """x [T, heads, d], neighbouring pairs turned; angle [T, d / 2]."""
    c, s = torch.cos(angle).unsqueeze(1), torch.sin(angle).unsqueeze(1)
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * c - v * s, v * c + u * s], -1).reshape(x.shape)


def _attention(q, k, v, scale, window=0, sink=False):
    """q [T, H, d], k [T, G, d], v [T, G, dv] -> [T, H, dv], causal; with a window the last `window` positions; sink: one more 1 below."""
    T, H, G = q.shape[0], q.shape[1], k.shape[1]
    far = torch.arange(T, device="cuda").unsqueeze(1) - torch.arange(T, device="cuda")
    hidden = (far < 0) | (far >= window if window else far < 0)
    out = torch.empty(T, H, v.shape[2], dtype=F64, device="cuda")
    for h in range(H):
        g = h // (H // G)
        s = (q[:, h].contiguous() @ k[:, g].t().contiguous() * scale).masked_fill_(hidden, -math.inf)
        m = s.amax(1, keepdim=True)
        m = m.clamp(min=0.0) if sink else m
        p = torch.exp(s - m)
        out[:, h] = (p @ v[:, g].contiguous()) / (p.sum(1, keepdim=True) + (torch.exp(-m) if sink else 0.0))
    return out


TQ_CENTERS = {2: (0.4528427, 1.5102326), 3: (0.2453404, 0.7561303, 1.3441838, 2.1521645)}
TQ_EDGES = {2: (0.98153765,), 3: (0.50073535, 1.05015705, 1.74817415)}


def _compressed(x, signs, bits):
    """What the compressed cache gives back of rows x [T, heads, d]: signs, Walsh-Hadamard rotation, the nearest of 2^bits centers, and back."""
    d = x.shape[-1]
    H = torch.ones(1, 1, dtype=F64, device="cuda")
    while H.shape[0] < d:
        H = torch.cat([torch.cat([H, H], 1), torch.cat([H, -H], 1)], 0)
    H = H / math.sqrt(d)
    r = (x * signs) @ H
    edges = torch.tensor([-e for e in reversed(TQ_EDGES[bits])] + [0.0] + list(TQ_EDGES[bits]), dtype=F64, device="cuda") / math.sqrt(d)
    centers = torch.tensor([-c for c in reversed(TQ_CENTERS[bits])] + list(TQ_CENTERS[bits]), dtype=F64, device="cuda") / math.sqrt(d)
    return (centers[torch.bucketize(r.contiguous(), edges, right=True)] @ H) * signs


def _gguf_exact(case, seed, sequences, want):
    """Logits after the places want[s] of the token sequences s, each [len(want[s]), vocab]."""
    model = _gguf_model(case, seed)
    c, w = model.config, _Gguf(model)
    D, H, G = c.head_dim, c.num_heads, c.num_kv_heads
    signs = _signs(case, c, seed)
    lens = [len(s) for s in sequences]
    ids = torch.from_numpy(np.concatenate(sequences).astype(np.int64)).cuda()
    pos = torch.cat([torch.arange(n, device="cuda") for n in lens])
    # angles as the model defines them: frequencies and their products with the position are 32-bit numbers
    freq = 1.0 / torch.pow(torch.tensor(c.rope_freq_base, dtype=F64), torch.arange(0, D, 2, dtype=F64) / D)
    angle = (pos.float().unsqueeze(1) * freq.float().cuda()).to(F64)
    x = w.matrix("token_embd.weight")[ids].clone()
    for i in range(c.num_layers):
        p = f"blk.{i}."
        h = _rms(x, c.norm_eps) * w.matrix(p + "attn_norm.weight")
        q = _turn_pairs((h @ w.matrix(p + "attn_q.weight").t()).view(-1, H, D), angle)
        k = _turn_pairs((h @ w.matrix(p + "attn_k.weight").t()).view(-1, G, D), angle)
        v = (h @ w.matrix(p + "attn_v.weight").t()).view(-1, G, D)
        if signs is not None:
            sg = torch.from_numpy(signs[i]).cuda().to(F64)
            k, v = _compressed(k, sg[:, 0], int(case["kv"][2])), _compressed(v, sg[:, 1], int(case["kv"][2]))
        a, at = torch.empty(len(ids), H * D, dtype=F64, device="cuda"), 0
        for n in lens:
            a[at:at + n] = _attention(q[at:at + n], k[at:at + n], v[at:at + n], D ** -0.5).reshape(n, -1)
            at += n
        x = x + a @ w.matrix(p + "attn_output.weight").t()
        h = _rms(x, c.norm_eps) * w.matrix(p + "ffn_norm.weight")
        ff = lambda y, gate, up, down: (torch.nn.functional.silu(y @ gate.t()) * (y @ up.t())) @ down.t()
        if not c.num_experts:
            x = x + ff(h, *(w.matrix(p + f"ffn_{n}.weight") for n in ("gate", "up", "down")))
            continue
        best, which = torch.topk(h @ w.matrix(p + "ffn_gate_inp.weight").t(), c.num_experts_per_token, dim=1)
        share = torch.softmax(best, 1)
        for e in range(c.num_experts):
            rows, slot = torch.nonzero(which == e, as_tuple=True)
            if len(rows):
                x[rows] += share[rows, slot].unsqueeze(1) * ff(h[rows], *(w.matrix(p + f"ffn_{n}_exps.weight", e) for n in ("gate", "up", "down")))
    starts = np.concatenate([[0], np.cumsum(lens)[:-1]])
    rows = torch.tensor([int(o) + t for o, places in zip(starts, want) for t in places], device="cuda")
    head = w.matrix("output.weight").t()
    logits = (_rms(x[rows], c.norm_eps) * w.matrix("output_norm.weight")) @ head
    return torch.split(logits.cpu(), [len(p) for p in want])


def _layer_norm(x, w, eps):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * w


def _frequencies(rot):
    """(angle of a position per pair, factor on cosine and sine), with the blend of a scaled rotation."""
    n = rot["dims"]
    f = torch.tensor([rot["base"] ** (-2.0 * i / n) for i in range(n // 2)], dtype=F64, device="cuda")
    sc = rot.get("scaling")
    if not sc:
        return f, 1.0
    at = lambda t: n * math.log(sc["original"] / (2 * math.pi * t)) / (2 * math.log(rot["base"]))
    lo, hi = max(math.floor(at(sc["fast"])), 0), min(math.ceil(at(sc["slow"])), n - 1)
    ramp = ((torch.arange(n // 2, dtype=F64, device="cuda") - lo) / max(hi - lo, 0.001)).clamp(0.0, 1.0)
    return f / sc["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(sc["factor"]) + 1.0


def _rotated(x, rot, halves=False):
    """x [T, heads, d], all values rotated: neighbouring pairs, or value i with value i + d / 2."""
    f, mag = _frequencies(rot)
    a = torch.arange(len(x), dtype=F64, device="cuda").unsqueeze(1) * f
    if not halves:
        return _turn_pairs(x, a) * mag
    c, s, n = torch.cos(a).unsqueeze(1), torch.sin(a).unsqueeze(1), x.shape[-1] // 2
    return torch.cat([x[..., :n] * c - x[..., n:] * s, x[..., n:] * c + x[..., :n] * s], -1) * mag


def _latent(h, w, mx, eps, queries, halves):
    """Attention over keys and values expanded from a latent; keys carry a rotated part that all heads share.  -> [T, heads, vdim]"""
    T, H, d, kr = len(h), mx["heads"], mx["dim"], mx["kv_rank"]
    q, dkv = queries.view(T, H, -1), h @ w("dkv").t()
    c = _rms(dkv[:, :kr], eps) * w("dkv.norm")
    k_rot = _rotated(dkv[:, kr:].unsqueeze(1), mx["rot"], halves).expand(T, H, -1)
    q = torch.cat([q[..., :d], _rotated(q[..., d:], mx["rot"], halves)], -1)
    k = torch.cat([(c @ w("uk").t()).view(T, H, d), k_rot], -1)
    return _attention(q, k, (c @ w("uv").t()).view(T, H, -1), mx["scale"], mx.get("mask", {"size": 0})["size"])


def _mlstm(h, w, mx, eps):
    """The matrix memory, one token after the other, all heads at once."""
    T, H, d, cap = len(h), mx["heads"], mx["dim"], mx["gate_cap"]
    q, k = (h @ w("q").t()).view(T, H, d) * d ** -0.5, (h @ w("k").t()).view(T, H, d)
    v = (h @ w("v").t()).view(T, H, -1)
    li = cap * torch.tanh((h @ w("i").t() + w("i.b")) / cap)
    lf = torch.nn.functional.logsigmoid(cap * torch.tanh((h @ w("f").t() + w("f.b")) / cap))
    S, n, m = torch.zeros(H, d, v.shape[2], dtype=F64, device="cuda"), torch.zeros(H, d, dtype=F64, device="cuda"), torch.zeros(H, dtype=F64, device="cuda")
    out = torch.empty_like(v)
    for t in range(T):
        m2 = torch.maximum(lf[t] + m, li[t])
        a, b, m = torch.exp(lf[t] + m - m2).view(H, 1), torch.exp(li[t] - m2).view(H, 1), m2
        S = a.unsqueeze(2) * S + (b * k[t]).unsqueeze(2) * v[t].unsqueeze(1)
        n = a * n + b * k[t]
        top = (S * q[t].unsqueeze(2)).sum(1)
        out[t] = top / (torch.maximum((n * q[t]).sum(1).abs(), torch.exp(-m)) + 1e-6).unsqueeze(1)
    return (_rms(out, eps).reshape(T, -1) * w("norm") * torch.sigmoid(h @ w("g").t())) @ w("o").t()


def _delta(h, w, mx, eps):
    """The delta rule, one token after the other, all heads at once."""
    T, H, G, d = len(h), mx["heads"], mx["kv_heads"], mx["dim"]

    def short(name):                                                            # projection, causal convolution per channel, silu
        y, f = h @ w(name).t(), w(name + ".conv")
        z = torch.zeros_like(y)
        for j in range(f.shape[1]):
            back = f.shape[1] - 1 - j
            z[back:] += f[:, j] * (y[:T - back] if back else y)
        return torch.nn.functional.silu(z)
    unit = lambda u: u / torch.sqrt((u * u).sum(-1, keepdim=True) + 1e-6)
    spread = lambda u: u.repeat_interleave(H // G, 1)
    q, k = spread(unit(short("q").view(T, G, d))) * d ** -0.5, spread(unit(short("k").view(T, G, d)))
    v = short("v").view(T, H, -1)
    beta = torch.sigmoid(h @ w("b").t())
    g = torch.exp(-torch.exp(w("A_log")) * torch.nn.functional.softplus(h @ w("a").t() + w("dt_bias")))
    S, out = torch.zeros(H, d, v.shape[2], dtype=F64, device="cuda"), torch.empty_like(v)
    for t in range(T):
        S = g[t].view(H, 1, 1) * S
        u = beta[t].unsqueeze(1) * (v[t] - (S * k[t].unsqueeze(2)).sum(1))
        S = S + k[t].unsqueeze(2) * u.unsqueeze(1)
        out[t] = (S * q[t].unsqueeze(2)).sum(1)
    return ((_rms(out, eps) * w("norm")).reshape(T, -1) * torch.nn.functional.silu(h @ w("g").t())) @ w("o").t()


def _layered_exact(case, seed):
    cfg, src = _layered_config(case), _Layered(seed)
    shapes = dict(lg.layered_model.parse_config(cfg).tensor_shapes())           # names and sizes only
    W = lambda name: src.tensor(name, shapes[name]).to(F64)
    ids = torch.from_numpy(np.concatenate([_ids(case, seed, case["prompt"]), _ids(case, seed, case["steps"], 1)]).astype(np.int64)).cuda()
    T, eps, first, kvs = len(ids), cfg["norm"]["eps"], case["prompt"] - 1, {}
    x = W("embed")[ids]
    if case["design"] == "Zamelix":
        big = cfg["embedding"]["bigram"]
        row = torch.full_like(ids, big["buckets"])
        row[1:] = (ids[:-1] * big["mul_prev"] + ids[1:] * big["mul_cur"]) % big["buckets"]
        x = x + W("bigram")[row]
    for i, lay in enumerate(cfg["layers"]):
        p, mx = f"l{i}.", lay["mixer"]
        w, f = (lambda n: W(p + "mix." + n)), (lambda n: W(p + "mlp." + n).t())
        if case["design"] == "Zamelix":
            if lay["type"] == "mlstm":
                y = _mlstm(x, w, mx, eps)
            else:
                y = _latent(x, w, mx, eps, x @ w("q").t(), False) * torch.sigmoid(x @ w("g").t()).unsqueeze(2)
                y = y.reshape(T, -1) @ w("o").t()
            x = x + cfg["residual_mult"] * _layer_norm(y, W(p + "norm1"), eps)
            if lay["mlp"]:
                y = (torch.nn.functional.gelu(x @ f("gate"), approximate="tanh") * (x @ f("up"))) @ f("down")
                x = x + cfg["residual_mult"] * _layer_norm(y, W(p + "norm2"), eps)
            continue
        h = _layer_norm(x, W(p + "norm1"), eps)
        if lay["type"] == "delta":
            y = _delta(h, w, mx, eps)
        elif lay["type"] == "attention":
            if "kv_from" not in mx:
                k = _rotated((h @ w("k").t() + w("k.b")).view(T, mx["kv_heads"], -1), mx["rot"])
                kvs[i] = k, (h @ w("v").t() + w("v.b")).view(T, mx["kv_heads"], -1)
            q = _rotated((h @ w("q").t() + w("q.b")).view(T, mx["heads"], -1), mx["rot"])
            y = _attention(q, *kvs[mx.get("kv_from", i)], mx["scale"], mx["mask"]["size"], sink=True)
            y = y.reshape(T, -1) @ w("o").t() + w("o.b")
        else:
            queries = (_rms(h @ w("dq").t(), eps) * w("dq.norm")) @ w("uq").t()
            y = (_latent(h, w, mx, eps, queries, True).reshape(T, -1) * torch.sigmoid(h @ w("g").t())) @ w("o").t()
        x = x + _layer_norm(y, W(p + "norm1b"), eps) * W(p + "ls1")
        y = (torch.relu(_layer_norm(x, W(p + "norm2"), eps) @ f("up")) ** 2) @ f("down")
        x = x + _layer_norm(y, W(p + "norm2b"), eps) * W(p + "ls2")
    logits = _layer_norm(x[first:], W("final.norm"), eps) @ W("head").t()
    if case["design"] == "Tarudra":
        logits = cfg["logit_softcap"] * torch.tanh(logits / cfg["logit_softcap"])
    return logits.cpu()


def exact(case, seed):
    if case["kind"] == "generate":
        rows = _layered_exact(case, seed)
        return [rows[:1]] + [rows[i] for i in range(1, len(rows))]
    if case["kind"] == "prompt":
        return _gguf_exact(case, seed, [_ids(case, seed, case["tokens"])], [[case["tokens"] - 1]])[0]
    if case["kind"] == "decode":
        n = case["context"]
        ids = np.concatenate([_ids(case, seed, n), _ids(case, seed, case["steps"], 1)])
        return list(_gguf_exact(case, seed, [ids], [list(range(n, n + case["steps"]))])[0])
    lens = _lengths(case, seed)
    after = _ids(case, seed, case["steps"] * case["sequences"], 1).reshape(case["steps"], -1)
    got = _gguf_exact(case, seed, [np.concatenate([_ids(case, seed, n, 10 + s), after[:, s]]) for s, n in enumerate(lens)],
                      [list(range(n, n + case["steps"])) for n in lens])
    return [torch.stack([got[s][t] for s in range(len(lens))]) for t in range(case["steps"])]
