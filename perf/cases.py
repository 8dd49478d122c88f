"""The work that a user of the serving engine has it do, as cases with sizes, data and expected results.

A case is one request (or one step of several requests) of a loaded model, through the runner that the server
drives: the first token of a prompt, a reply of some tokens after a cached conversation, several sequences decoded
together, an image turned into embedding rows. Models have the layer widths of this repository's presets and
benchmark sizes with fewer layers (every layer of a model is alike, so depth only repeats the work); one case has a
preset's full depth.

Weights are random, drawn in the quantised formats themselves; what a trained model has and plain noise lacks is
built in where it matters: a next token that stands out (every token has one successor, whose head row points at
that token's embedding, so that sampled tokens do not hang on the last bits of a logit) and routers that know their
tokens' experts (router rows are sums of the embeddings of the tokens in use). Residual projections are scaled by
the depth.
"""
from __future__ import annotations

import json
import math
import os
import shutil
import tempfile

import numpy as np
import torch

VOCAB = 32000
USED = 512          # distinct tokens that prompts are made of
F64 = torch.float64

# layer widths of the presets: width, heads, key/value heads, feed-forward, experts, experts per token
SHAPES = {
    "llama2-7b": (4096, 32, 32, 11008, 0, 0),
    "llama2-13b": (5120, 40, 40, 13824, 0, 0),
    "mistral-7b": (4096, 32, 8, 14336, 0, 0),
    "orca-mini-3b": (3200, 32, 32, 8640, 0, 0),    # head size 100; rows that are no multiple of 256
    "mixtral-8x7b": (4096, 32, 8, 14336, 8, 2),
}
ROPE_BASE = {"mistral-7b": 1e6, "mixtral-8x7b": 1e6}
# layer-list models at the sizes that the benchmark uses: width, layers (a = attention, r = retention), heads,
# key/value heads, head size, expert feed-forward, experts, per token, shared feed-forward, retention heads, dim, vdim
STACKS = {
    "bizulix-s": (1024, "aaaraaar", 16, 4, 64, 512, 8, 2, 1024, (8, 64, 128)),
    "bizulix-m": (2048, "aaar", 16, 4, 128, 1024, 8, 2, 2048, (16, 64, 128)),
}
FTYPES = {"Q4_0": 2, "Q8_0": 7, "Q4_K_M": 15, "Q5_K_M": 17}         # GGUF general.file_type
GGML = {"F32": 0, "F16": 1, "Q4_0": 2, "Q8_0": 8, "Q4_K": 12, "Q5_K": 13, "Q6_K": 14}
BLOCK = {"Q4_0": (32, 18), "Q8_0": (32, 34), "Q4_K": (256, 144), "Q5_K": (256, 176), "Q6_K": (256, 210)}
CLIP = dict(E=1024, F=4096, heads=16, patch=14, out=4096)           # ViT-L/14, projected to a 4096-wide model


def listed() -> list[dict]:
    return [
        # the headline: one user's chat turn on the full Llama-2-7B, the conversation already cached; latency per token
        dict(name="reply-7b-full", kind="reply", model="llama2-7b", ftype="Q4_K_M", layers=32, prompt=129, tokens=33),
        # the same far into a conversation, grouped key/value heads, a smaller file type
        dict(name="reply-long", kind="reply", model="mistral-7b", ftype="Q4_0", layers=8, prompt=3400, tokens=17),
        # several users at once: the server's default of four, and a full house of sixteen
        dict(name="batch-4", kind="batch", model="llama2-7b", ftype="Q4_K_M", layers=8, prompt=200, tokens=17, rows=4),
        dict(name="batch-16", kind="batch", model="mistral-7b", ftype="Q8_0", layers=4, prompt=333, tokens=17, rows=16),
        # time to the first token: a short question, an ordinary prompt, a pasted document
        dict(name="prompt-33", kind="prompt", model="llama2-7b", ftype="Q4_K_M", layers=8, prompt=33, tokens=1),
        dict(name="prompt-509", kind="prompt", model="mistral-7b", ftype="Q5_K_M", layers=6, prompt=509, tokens=1),
        dict(name="prompt-2048", kind="prompt", model="llama2-7b", ftype="Q4_K_M", layers=8, prompt=2048, tokens=1),
        # routed experts: an ordinary prompt, and four users' replies
        dict(name="experts-prompt", kind="prompt", model="mixtral-8x7b", ftype="Q4_K_M", layers=2, prompt=1000, tokens=1),
        dict(name="experts-batch-4", kind="batch", model="mixtral-8x7b", ftype="Q4_K_M", layers=2, prompt=200, tokens=17, rows=4),
        # layer-list models in bfloat16: a document, and a short question with its reply (launches and latency)
        dict(name="stack-prompt", kind="prompt", model="bizulix-m", ftype="bf16", layers=4, prompt=2048, tokens=1),
        dict(name="stack-reply", kind="reply", model="bizulix-s", ftype="bf16", layers=8, prompt=61, tokens=33),
        # a picture in a prompt: the vision tower and its projector
        dict(name="image-336", kind="image", size=336, layers=23),
    ]


def draw(rng) -> dict:
    def log(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    kind = rng.choice(["prompt", "prompt", "prompt", "reply", "reply", "batch", "batch", "image"])
    if kind == "image":
        return dict(kind="image", size=rng.choice([224, 280, 336]), layers=rng.randint(6, 23))
    family = rng.choice(["dense", "dense", "dense", "experts", "stack", "stack"])
    if family == "dense":
        model = rng.choice(["llama2-7b", "llama2-13b", "mistral-7b", "orca-mini-3b"])
        ftype = rng.choice(["Q4_0", "Q8_0"] if model == "orca-mini-3b" else list(FTYPES))
        layers = rng.randint(2, 6)
    elif family == "experts":
        model, ftype, layers = "mixtral-8x7b", rng.choice(["Q4_0", "Q4_K_M"]), rng.randint(1, 2)
    else:
        model = rng.choice(list(STACKS))
        ftype, layers = rng.choice(["bf16", "bf16", "f32"]), len(STACKS[model][1])
    longest = 1000 if family == "experts" or ftype == "f32" else 2048
    c = dict(kind=kind, model=model, ftype=ftype, layers=layers, tokens=1)
    if kind == "prompt":
        c.update(prompt=log(8, longest))
    elif kind == "reply":
        c.update(prompt=log(16, 400 if family == "stack" else 1900 if model == "orca-mini-3b" else 3400), tokens=rng.randint(9, 33))
    else:
        c.update(prompt=log(16, 120 if family == "stack" else 500), tokens=rng.randint(9, 17), rows=rng.randint(2, 16))
    return c


# ---------------------------------------------------------------------------------------------- random numbers
def _gen(*key) -> torch.Generator:
    x = 0x9E3779B97F4A7C15
    for k in key:
        x = ((x ^ (int(k) + 0x632BE59BD9B4E019)) * 0xD1342543DE82EF95) % (1 << 64)
        x ^= x >> 29
    g = torch.Generator(device="cuda")
    g.manual_seed(x % (1 << 62))
    return g


def _tokens(seed: int) -> tuple[torch.Tensor, torch.Tensor]:
    """The tokens in use, in the order in which each is followed by the next (a ring), and that map."""
    ids = torch.randperm(VOCAB - 3, generator=_gen(seed, 1), device="cuda")[:USED] + 3
    return ids, torch.roll(ids, -1)


def _prompts(case: dict, seed: int) -> list[list[int]]:
    ids, _ = _tokens(seed)
    rows, out = case.get("rows", 1), []
    for r in range(rows):
        n = case["prompt"] if rows == 1 else max(2, case["prompt"] * (2 + r % 3) // 3)  # users' prompts differ in length
        at = torch.randint(0, USED, (n,), generator=_gen(seed, 2, r), device="cuda")
        out.append(ids[at].tolist())
    return out


def _replies(case: dict, seed: int) -> list[list[int]]:
    """What follows each prompt: the ring from its last token on."""
    ids, _ = _tokens(seed)
    ids = ids.tolist()
    place = {t: i for i, t in enumerate(ids)}
    return [[ids[(place[p[-1]] + 1 + j) % USED] for j in range(case["tokens"])] for p in _prompts(case, seed)]


# ---------------------------------------------------------------------------------------------- quantised blocks
def _f16(x: torch.Tensor) -> torch.Tensor:
    return x.to(torch.float16).view(torch.uint8).reshape(-1, 2)


def _pack6(sc: torch.Tensor, m: torch.Tensor) -> torch.Tensor:
    """Eight 6-bit scales and minima in twelve bytes, as Q4_K and Q5_K blocks hold them."""
    a = sc[:, :4] | ((sc[:, 4:] >> 4) << 6)
    b = m[:, :4] | ((m[:, 4:] >> 4) << 6)
    c = (sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)
    return torch.cat([a, b, c], 1).to(torch.uint8)


def _random_blocks(kind: str, rows: int, K: int, std: float, g) -> torch.Tensor:
    """[blocks, bytes] of random weights with about this standard deviation."""
    blk, nb = BLOCK[kind]
    n = rows * K // blk
    out = torch.randint(0, 256, (n, nb), dtype=torch.uint8, device="cuda", generator=g)
    u = 0.75 + 0.5 * torch.rand(n, device="cuda", generator=g)
    if kind in ("Q4_0", "Q8_0"):
        if kind == "Q4_0":                                 # codes 1 .. 15: no common offset of all weights
            q = torch.randint(1, 16, (2, n, 16), dtype=torch.uint8, device="cuda", generator=g)
            out[:, 2:] = q[0] | (q[1] << 4)
        out[:, :2] = _f16(u * (std / (4.6 if kind == "Q4_0" else 73.0)))
    elif kind == "Q6_K":
        out[:, 192:208] = torch.randint(64, 128, (n, 16), dtype=torch.uint8, device="cuda", generator=g)
        out[:, 208:] = _f16(u * (std / 18.5 / 96.0))
    else:
        q_std, mid = (4.6, 7.5) if kind == "Q4_K" else (9.2, 15.5)
        d = u * (std / q_std / 47.0)
        sc = torch.randint(32, 64, (n, 8), dtype=torch.int32, device="cuda", generator=g)
        out[:, :2], out[:, 2:4] = _f16(d), _f16(d * mid * 64.0 / 63.0)
        out[:, 4:16] = _pack6(sc, (sc * 63 + 32) // 64)   # minima that centre the weights near zero
    return out


def _quantise(kind: str, x: torch.Tensor) -> torch.Tensor:
    """[rows, K] floats -> blocks, by plain rounding (the output matrix)."""
    if kind == "Q8_0":
        b = x.reshape(-1, 32).float()
        d = (b.abs().amax(1) / 127.0).to(torch.float16)
        q = (b / d.float().clamp_min(1e-12)[:, None]).round().clamp(-127, 127).to(torch.int8)
        return torch.cat([d.view(torch.uint8).reshape(-1, 2), q.view(torch.uint8)], 1)
    b = x.reshape(-1, 16, 16).float()
    s = b.abs().amax(2) / 31.0
    d = (s.amax(1) / 127.0).to(torch.float16)
    sc = (s / d.float().clamp_min(1e-12)[:, None]).round().clamp(1, 127)
    q = ((b / (sc * d.float()[:, None]).clamp_min(1e-12)[..., None]).round().clamp(-32, 31) + 32).to(torch.uint8).reshape(-1, 2, 4, 32)
    ql = torch.cat([(q[:, :, 0] & 15) | ((q[:, :, 2] & 15) << 4), (q[:, :, 1] & 15) | ((q[:, :, 3] & 15) << 4)], 2)
    qh = (q[:, :, 0] >> 4) | ((q[:, :, 1] >> 4) << 2) | ((q[:, :, 2] >> 4) << 4) | ((q[:, :, 3] >> 4) << 6)
    return torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.uint8), d.view(torch.uint8).reshape(-1, 2)], 1)


def _values(kind: str, b: torch.Tensor, rows: int) -> torch.Tensor:
    """Blocks -> [rows, K] in float64, by the formats' definitions."""
    half = lambda at: b[:, at:at + 2].contiguous().view(torch.float16).to(F64)  # noqa: E731  [blocks, 1]
    if kind == "Q4_0":
        q = b[:, 2:]
        w = (torch.cat([q & 15, q >> 4], 1).to(F64) - 8.0) * half(0)
    elif kind == "Q8_0":
        w = b[:, 2:].contiguous().view(torch.int8).to(F64) * half(0)
    elif kind == "Q6_K":
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
        q = torch.stack([(ql[:, :, 0] & 15) | ((qh & 3) << 4), (ql[:, :, 1] & 15) | (((qh >> 2) & 3) << 4),
                         (ql[:, :, 0] >> 4) | (((qh >> 4) & 3) << 4), (ql[:, :, 1] >> 4) | ((qh >> 6) << 4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).to(F64) * half(208)
        w = (q.reshape(-1, 16, 16).to(F64) - 32.0) * sc[..., None]
    else:
        s = b[:, 4:16].to(torch.int32)
        sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | ((s[:, :4] >> 6) << 4)], 1).to(F64) * half(0)
        m = torch.cat([s[:, 4:8] & 63, (s[:, 8:] >> 4) | ((s[:, 4:8] >> 6) << 4)], 1).to(F64) * half(2)
        qs = b[:, 16 if kind == "Q4_K" else 48:].reshape(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).reshape(-1, 8, 32).to(F64)
        if kind == "Q5_K":
            bit = torch.arange(8, device=b.device, dtype=torch.uint8)[None, :, None]
            q = q + 16.0 * ((b[:, 16:48][:, None] >> bit) & 1).to(F64)
        w = q * sc[..., None] - m[..., None]
    return w.reshape(rows, -1)


# ---------------------------------------------------------------------------------------------- GGUF models
def _dims(case: dict) -> dict:
    E, H, G, F, X, top = SHAPES[case["model"]]
    return dict(E=E, H=H, G=G, D=E // H, F=F, X=X, top=top, L=case["layers"])


def _kind(ftype: str, role: str, layer: int, L: int, K: int) -> str:
    """Block format of a matrix in a file of this type (the public mix of the K-quant files)."""
    if K % 256:
        return "Q8_0" if role == "output" or ftype == "Q8_0" else "Q4_0"
    if ftype == "Q8_0":
        return "Q8_0"
    more = layer < L // 8 or layer >= 7 * L // 8 or (layer - L // 8) % 3 == 2
    if role == "output" or (ftype != "Q4_0" and role in ("v", "down") and more):
        return "Q6_K"
    return {"Q4_0": "Q4_0", "Q4_K_M": "Q4_K", "Q5_K_M": "Q5_K"}[ftype]


class _Gguf:
    """The matrices of a case's model: blocks by name, made when asked for."""

    def __init__(self, case: dict, seed: int):
        self.case, self.seed, self.d = case, seed, _dims(case)
        d, ft = self.d, case["ftype"]
        self.mats = {"token_embd": (_kind(ft, "embd", 0, d["L"], d["E"]), VOCAB, d["E"], 1.0)}
        res = (2.0 * d["L"]) ** -0.5
        for i in range(d["L"]):
            def add(name, role, rows, K, gain, n=1, i=i):
                self.mats[f"blk.{i}.{name}"] = (_kind(ft, role, i, d["L"], K), rows * n, K, gain * K ** -0.5)
            add("attn_q", "q", d["E"], d["E"], 1.0)
            add("attn_k", "k", d["G"] * d["D"], d["E"], 1.0)
            add("attn_v", "v", d["G"] * d["D"], d["E"], 1.0)
            add("attn_output", "o", d["E"], d["E"], res)
            x, n = ("_exps", d["X"]) if d["X"] else ("", 1)
            add("ffn_gate" + x, "gate", d["F"], d["E"], 1.0, n)
            add("ffn_up" + x, "up", d["F"], d["E"], 1.0, n)
            add("ffn_down" + x, "down", d["E"], d["F"], 2.0 * res, n)
        self.mats["output"] = (_kind(ft, "output", 0, d["L"], d["E"]), VOCAB, d["E"], 0.0)
        self.names = list(self.mats)

    def blocks(self, name: str) -> torch.Tensor:
        kind, rows, K, std = self.mats[name]
        g = _gen(self.seed, 3, self.names.index(name))
        if name != "output":
            return _random_blocks(kind, rows, K, std, g)
        e = self.values("token_embd").float()     # a token's successor answers to its embedding; the rest is noise
        w = torch.randn(rows, K, device="cuda", generator=g)
        ids, nxt = _tokens(self.seed)
        w[nxt] = e[ids]
        return _quantise(kind, w * (28.0 / K))

    def values(self, name: str) -> torch.Tensor:
        return _values(self.mats[name][0], self.blocks(name), self.mats[name][1])

    def vector(self, i: int) -> torch.Tensor:
        """Norm weights: 2 * layer (+ 1 for the feed-forward's), the final one at 2 * layers."""
        return 1.0 + 0.05 * torch.randn(self.d["E"], device="cuda", generator=_gen(self.seed, 4, i))

    def router(self, i: int) -> torch.Tensor:
        e = self.values("token_embd")[_tokens(self.seed)[0]].float()
        return _router(e, self.d["X"], self.d["top"], _gen(self.seed, 5, i))


def _router(e: torch.Tensor, X: int, top: int, g) -> torch.Tensor:
    """[X, E]: every token in use has `top` experts of its own, whose rows hold its embedding."""
    pick = torch.rand(e.shape[0], X, device="cuda", generator=g).argsort(1)[:, :top]
    on = torch.zeros(e.shape[0], X, device="cuda").scatter_(1, pick, 1.0)
    return (on.T @ e) * (4.0 / e.shape[1])


def _scratch_dir(need: int) -> str:
    shm = "/dev/shm"
    room = shutil.disk_usage(shm).free if os.path.isdir(shm) and os.access(shm, os.W_OK) else 0
    return tempfile.mkdtemp(prefix="omx_cases_", dir=shm if room > 2 * need else None)


def _gguf_runner(case: dict, seed: int):
    from ollama_operator_amd.engine.runner import Runner
    from ollama_operator_amd.gguf.constants import GGMLType
    from ollama_operator_amd.gguf.writer import GGUFWriter
    from ollama_operator_amd.models.config import ModelConfig
    m, d, rows = _Gguf(case, seed), _dims(case), case.get("rows", 1)
    cfg = ModelConfig(name=case["model"], n_vocab=VOCAB, n_embd=d["E"], n_layer=d["L"], n_head=d["H"], n_head_kv=d["G"], n_ff=d["F"],
                      n_rot=d["D"], rope_base=ROPE_BASE.get(case["model"], 1e4), ctx_len=4096, n_expert=d["X"], n_expert_used=d["top"])
    folder = _scratch_dir(int(_weight_bytes(case)[1]))
    try:
        path = os.path.join(folder, "model.gguf")
        w = GGUFWriter(path)
        for k, v in cfg.to_gguf_metadata().items():
            w.add(k, v)
        w.add("llama.vocab_size", VOCAB)
        w.add("general.file_type", FTYPES[case["ftype"]])
        for name, (kind, n, K, _std) in m.mats.items():
            shape = (K, n // d["X"], d["X"]) if name.endswith("_exps") else (K, n)
            w.add_tensor(name + ".weight", shape, GGMLType(GGML[kind]), lambda name=name: m.blocks(name).cpu().numpy())
        vec = lambda t: (lambda: t.float().cpu().numpy())  # noqa: E731
        for i in range(d["L"]):
            w.add_tensor(f"blk.{i}.attn_norm.weight", (d["E"],), GGMLType.F32, vec(m.vector(2 * i)))
            w.add_tensor(f"blk.{i}.ffn_norm.weight", (d["E"],), GGMLType.F32, vec(m.vector(2 * i + 1)))
            if d["X"]:
                w.add_tensor(f"blk.{i}.ffn_gate_inp.weight", (d["E"], d["X"]), GGMLType.F32, vec(m.router(i)))
        w.add_tensor("output_norm.weight", (d["E"],), GGMLType.F32, vec(m.vector(2 * d["L"])))
        w.write()
        return Runner(path, device="cuda:0", max_batch=2048, max_seqs=rows, ctx=4096)
    finally:
        shutil.rmtree(folder, ignore_errors=True)


def _rope(x: torch.Tensor, base: float) -> torch.Tensor:
    """x [n, heads, D]: dimensions 2i and 2i + 1 are turned by position * base^(-2i / D)."""
    n, _, D = x.shape
    f = (base ** (-torch.arange(0, D, 2, device=x.device, dtype=F64) / D)).float().to(F64)  # frequencies are 32-bit numbers
    a = torch.arange(n, device=x.device, dtype=F64)[:, None] * f
    c, s = torch.cos(a)[:, None], torch.sin(a)[:, None]
    u, v = x[..., 0::2], x[..., 1::2]
    return torch.stack([u * c - v * s, u * s + v * c], -1).reshape(x.shape)


def _softmax_attention(q, k, v, scale, cap=0.0, causal=True):
    """q [n, H, D], k / v [n, G, D]: grouped heads, one head at a time."""
    n, H, _ = q.shape
    r, out = H // k.shape[1], torch.empty(n, H, v.shape[2], dtype=F64, device=q.device)
    mask = torch.ones(n, n, dtype=torch.bool, device=q.device).triu(1)
    for h in range(H):
        s = (q[:, h] @ k[:, h // r].T) * scale
        if cap:
            s = cap * torch.tanh(s / cap)
        if causal:
            s = s.masked_fill_(mask, -math.inf)
        out[:, h] = torch.softmax(s, -1) @ v[:, h // r]
    return out.reshape(n, -1)


def _gguf_exact(case: dict, seed: int, seq: list[int]) -> torch.Tensor:
    m, d = _Gguf(case, seed), _dims(case)
    rms = lambda x, i: x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-5) * m.vector(i).to(F64)  # noqa: E731
    silu = torch.nn.functional.silu
    base = ROPE_BASE.get(case["model"], 1e4)
    x = m.values("token_embd")[torch.tensor(seq, device="cuda")]
    n = x.shape[0]
    for i in range(d["L"]):
        b = f"blk.{i}."
        h = rms(x, 2 * i)
        q = _rope((h @ m.values(b + "attn_q").T).view(n, d["H"], d["D"]), base)
        k = _rope((h @ m.values(b + "attn_k").T).view(n, d["G"], d["D"]), base)
        v = (h @ m.values(b + "attn_v").T).view(n, d["G"], d["D"])
        x = x + _softmax_attention(q, k, v, d["D"] ** -0.5) @ m.values(b + "attn_output").T
        h = rms(x, 2 * i + 1)
        if not d["X"]:
            x = x + (silu(h @ m.values(b + "ffn_gate").T) * (h @ m.values(b + "ffn_up").T)) @ m.values(b + "ffn_down").T
            continue
        val, idx = (h @ m.router(i).to(F64).T).topk(d["top"], -1)
        wt = torch.softmax(val, -1)
        gate, up, down = (m.values(b + f"ffn_{z}_exps").view(d["X"], -1, d["F"] if z == "down" else d["E"]) for z in ("gate", "up", "down"))
        y = torch.zeros_like(x)
        for e in range(d["X"]):
            t, j = (idx == e).nonzero(as_tuple=True)
            y[t] += wt[t, j][:, None] * ((silu(h[t] @ gate[e].T) * (h[t] @ up[e].T)) @ down[e].T)
        x = x + y
    return rms(x[-1:], 2 * d["L"]) @ m.values("output").T


# ---------------------------------------------------------------------------------------------- layer-list models
def _stack_config(case: dict) -> dict:
    E, pattern, H, G, D, F, X, top, Fs, (rh, rd, rv) = STACKS[case["model"]]
    layers = []
    for c in pattern:
        if c == "a":
            ent = dict(type="attention", mixer=dict(heads=H, kv_heads=G, dim=D, vdim=D, scale=D ** -0.5, softcap=50.0,
                                                    q_temp=dict(coef=0.1, every=1024)))
        else:
            ent = dict(type="retention", mixer=dict(heads=rh, dim=rd, vdim=rv, decay=[1.0 - 2.0 ** (-5 - i % 8) for i in range(rh)],
                                                    rot=dict(dims=rd, base=1e4)))
        ent["mlp"] = dict(kind="moe", router=dict(experts=X, top=top), expert=dict(ff=F), shared=dict(ff=Fs))
        layers.append(ent)
    return dict(architecture="Bizulix", vocab=VOCAB, width=E, layers=layers, norm=dict(eps=1e-6), residual_mult=1.0, logit_softcap=30.0)


def _stack_tensors(case: dict, seed: int) -> dict:
    E, pattern, H, G, D, F, X, top, Fs, (rh, rd, rv) = STACKS[case["model"]]
    g, T = _gen(seed, 6), {}

    def rnd(name, shape, s, mean=0.0):
        T[name] = (mean + s * torch.randn(*shape, device="cuda", generator=g)).to(torch.bfloat16)

    ids, nxt = _tokens(seed)
    res = (2.0 * len(pattern)) ** -0.5
    rnd("embed", (VOCAB, E), 1.0)
    for i, c in enumerate(pattern):
        p = f"l{i}."
        rnd(p + "norm1", (E,), 0.05, 1.0)
        rnd(p + "norm1.b", (E,), 0.05)
        nq, nk, nv, no = (H * D, G * D, G * D, H * D) if c == "a" else (rh * rd, rh * rd, rh * rv, rh * rv)
        for name, rows in (("q", nq), ("k", nk), ("v", nv)) + ((("g", no),) if c == "r" else ()):
            rnd(p + "mix." + name, (rows, E), E ** -0.5)
        rnd(p + "mix.o", (E, no), res * no ** -0.5)
        for e in ([f"e{e}" for e in range(X)] + ["shared"]):
            ff = Fs if e == "shared" else F
            rnd(f"{p}mlp.{e}.gate", (ff, E), E ** -0.5)
            rnd(f"{p}mlp.{e}.up", (ff, E), E ** -0.5)
            rnd(f"{p}mlp.{e}.down", (E, ff), res * ff ** -0.5)
        T[p + "mlp.router"] = _router(T["embed"][ids].float(), X, top, g).to(torch.bfloat16)
        rnd(p + "mlp.router.b", (X,), 0.05)
        rnd(p + "mlp.shared.sg", (1, E), E ** -0.5)
    rnd("final.norm", (E,), 0.05, 1.0)
    rnd("final.norm.b", (E,), 0.05)
    head = torch.randn(VOCAB, E, device="cuda", generator=g)
    head[nxt] = T["embed"][ids].float()
    T["head"] = (head * (28.0 / E)).to(torch.bfloat16)
    return T


def _stack_runner(case: dict, seed: int):
    from ollama_operator_amd.engine.safetensors_io import write_safetensors
    from ollama_operator_amd.engine.stack_runner import StackRunner
    folder = _scratch_dir(int(_weight_bytes(case)[1]))
    try:
        with open(os.path.join(folder, "config.json"), "w") as f:
            json.dump(_stack_config(case), f)
        write_safetensors(os.path.join(folder, "model.safetensors"), _stack_tensors(case, seed))
        return StackRunner(folder, device="cuda:0", max_batch=2048, max_seqs=max(2, case.get("rows", 1)), ctx=4096,
                           dtype={"bf16": "bfloat16", "f32": "float32"}[case["ftype"]])
    finally:
        shutil.rmtree(folder, ignore_errors=True)


def _stack_exact(case: dict, seed: int, seq: list[int]) -> torch.Tensor:
    E, pattern, H, G, D, F, X, top, Fs, (rh, rd, rv) = STACKS[case["model"]]
    T = _stack_tensors(case, seed)
    w = lambda name: T[name].to(F64)  # noqa: E731
    silu = torch.nn.functional.silu

    def norm(x, name):
        c = x - x.mean(-1, keepdim=True)
        return c * torch.rsqrt((c * c).mean(-1, keepdim=True) + 1e-6) * w(name) + w(name + ".b")

    def ff(h, p):
        return (silu(h @ w(p + ".gate").T) * (h @ w(p + ".up").T)) @ w(p + ".down").T

    x = w("embed")[torch.tensor(seq, device="cuda")]
    n = x.shape[0]
    at = torch.arange(n, device="cuda", dtype=F64)
    for i, c in enumerate(pattern):
        p = f"l{i}."
        h = norm(x, p + "norm1")
        q, k, v = (h @ w(p + "mix." + z).T for z in "qkv")
        if c == "a":
            q = q.view(n, H, D) * (1.0 + 0.1 * torch.log(torch.floor((at + 1) / 1024) + 1.0))[:, None, None]
            o = _softmax_attention(q, k.view(n, G, D), v.view(n, G, D), D ** -0.5, cap=50.0)
        else:
            def turn(z):
                f = 1e4 ** (-2.0 * torch.arange(rd // 2, device="cuda", dtype=F64) / rd)
                a = at[:, None] * f
                cs, sn = torch.cos(a)[:, None], torch.sin(a)[:, None]
                z = z.view(n, rh, rd)
                lo, hi = z[..., :rd // 2], z[..., rd // 2:]
                return torch.cat([lo * cs - hi * sn, hi * cs + lo * sn], -1)
            q, k, v = turn(q), turn(k) * rd ** -0.5, v.view(n, rh, rv)
            gap = (at[:, None] - at[None, :]).clamp_min(0.0)
            o = torch.empty(n, rh, rv, dtype=F64, device="cuda")
            for hd in range(rh):
                o[:, hd] = torch.tril((q[:, hd] @ k[:, hd].T) * (1.0 - 2.0 ** (-5 - hd % 8)) ** gap) @ v[:, hd]
            o = (o * torch.rsqrt((o * o).mean(-1, keepdim=True) + 1e-6)).reshape(n, -1) * silu(h @ w(p + "mix.g").T)
        y = o @ w(p + "mix.o").T
        val, idx = (h @ w(p + "mlp.router").T + w(p + "mlp.router.b")).topk(top, -1)
        wt = torch.softmax(val, -1)
        for e in range(X):
            t, j = (idx == e).nonzero(as_tuple=True)
            y[t] += wt[t, j][:, None] * ff(h[t], f"{p}mlp.e{e}")
        x = x + y + torch.sigmoid(h @ w(p + "mlp.shared.sg").T) * ff(h, p + "mlp.shared")
    return 30.0 * torch.tanh(norm(x[-1:], "final.norm") @ w("head").T / 30.0)


# ---------------------------------------------------------------------------------------------- images
def _clip_tensors(case: dict, seed: int):
    """(name, shape, 16-bit?, values) of a ViT with its two-layer projector."""
    E, F, out, p = CLIP["E"], CLIP["F"], CLIP["out"], CLIP["patch"]
    n_pos, g = (case["size"] // p) ** 2 + 1, _gen(seed, 7)

    def t(name, shape, std, half=True, mean=0.0):
        v = mean + std * torch.randn(*shape, device="cuda", generator=g)
        return name, shape, half, v.to(torch.float16 if half else torch.float32)

    yield t("v.patch_embd.weight", (E, 3, p, p), (3 * p * p) ** -0.5)
    yield t("v.class_embd", (E,), 0.5, False)
    yield t("v.position_embd.weight", (n_pos, E), 0.2)
    yield t("v.pre_ln.weight", (E,), 0.05, False, 1.0)
    yield t("v.pre_ln.bias", (E,), 0.02, False)
    res = (2.0 * case["layers"]) ** -0.5
    for i in range(case["layers"]):
        b = f"v.blk.{i}."
        for m, rows, K, gain in (("attn_q", E, E, 1.0), ("attn_k", E, E, 1.0), ("attn_v", E, E, 1.0), ("attn_out", E, E, res),
                                 ("ffn_up", F, E, 1.0), ("ffn_down", E, F, 2.0 * res)):
            yield t(b + m + ".weight", (rows, K), gain * K ** -0.5)
            yield t(b + m + ".bias", (rows,), 0.02, False)
        for ln in ("ln1", "ln2"):
            yield t(b + ln + ".weight", (E,), 0.05, False, 1.0)
            yield t(b + ln + ".bias", (E,), 0.02, False)
    for name, K in (("mm.0", E), ("mm.2", out)):
        yield t(name + ".weight", (out, K), K ** -0.5)
        yield t(name + ".bias", (out,), 0.02, False)


def _pixels(case: dict, seed: int) -> np.ndarray:
    """A picture as the preprocessor leaves it: smooth areas with some grain, normalised channels."""
    s = case["size"]
    rng = np.random.default_rng([seed, 8])
    coarse = torch.from_numpy(rng.standard_normal((1, 3, 9, 9)).astype(np.float32))
    px = torch.nn.functional.interpolate(coarse, size=(s, s), mode="bilinear", align_corners=True)[0].numpy()
    return np.ascontiguousarray(px + 0.1 * rng.standard_normal((3, s, s)).astype(np.float32))


def _clip_encoder(case: dict, seed: int):
    from ollama_operator_amd.gguf.constants import GGMLType
    from ollama_operator_amd.gguf.writer import GGUFWriter
    from ollama_operator_amd.models.clip import ClipEncoder
    folder = _scratch_dir(int(_weight_bytes(case)[1]))
    try:
        path = os.path.join(folder, "projector.gguf")
        w = GGUFWriter(path)
        v = "clip.vision."
        for k, x in {"general.architecture": "clip", "clip.has_vision_encoder": True, "clip.has_llava_projector": True,
                     "clip.projector_type": "mlp", "clip.use_gelu": False, v + "image_size": case["size"], v + "patch_size": CLIP["patch"],
                     v + "embedding_length": CLIP["E"], v + "feature_length": CLIP["F"], v + "block_count": case["layers"],
                     v + "attention.head_count": CLIP["heads"], v + "attention.layer_norm_epsilon": 1e-5}.items():
            w.add(k, x)
        for name, shape, half, x in _clip_tensors(case, seed):
            w.add_tensor(name, tuple(reversed(shape)), GGMLType.F16 if half else GGMLType.F32, x.cpu().numpy())
        w.write()
        return ClipEncoder(path, "cuda:0")
    finally:
        shutil.rmtree(folder, ignore_errors=True)


def _clip_exact(case: dict, seed: int) -> torch.Tensor:
    T = {name: x.to(F64) for name, _s, _h, x in _clip_tensors(case, seed)}
    E, H, p = CLIP["E"], CLIP["heads"], CLIP["patch"]
    g = case["size"] // p
    lin = lambda x, name: x @ T[name + ".weight"].T + T[name + ".bias"]  # noqa: E731
    ln = lambda x, name: torch.nn.functional.layer_norm(x, (E,), T[name + ".weight"], T[name + ".bias"], 1e-5)  # noqa: E731
    px = torch.from_numpy(_pixels(case, seed)).to("cuda", F64)
    x = px.reshape(3, g, p, g, p).permute(1, 3, 0, 2, 4).reshape(g * g, -1) @ T["v.patch_embd.weight"].reshape(E, -1).T
    x = ln(torch.cat([T["v.class_embd"][None], x]) + T["v.position_embd.weight"], "v.pre_ln")
    n = x.shape[0]
    for i in range(case["layers"]):
        b = f"v.blk.{i}."
        h = ln(x, b + "ln1")
        q, k, v = (lin(h, b + "attn_" + z).view(n, H, E // H) for z in "qkv")
        x = x + lin(_softmax_attention(q, k, v, (E // H) ** -0.5, causal=False), b + "attn_out")
        h = lin(ln(x, b + "ln2"), b + "ffn_up")
        x = x + lin(h * torch.sigmoid(1.702 * h), b + "ffn_down")
    return lin(torch.nn.functional.gelu(lin(x[1:], "mm.0")), "mm.2")


# ---------------------------------------------------------------------------------------------- the cases' interface
class _State(dict):
    """What a program keeps between calls; a model that is let go is closed, as the server closes one it unloads."""

    def __del__(self):
        if "runner" in self:
            self.pop("runner").close()


def prepare(case: dict, seed: int) -> dict:
    if case["kind"] == "image":
        return dict(case=case, encoder=_clip_encoder(case, seed), pixels=_pixels(case, seed))
    from ollama_operator_amd.engine.sampling import SamplingOptions
    r = _stack_runner(case, seed) if case["model"] in STACKS else _gguf_runner(case, seed)
    r.warmup()                                          # as the server does after a load
    rows = case.get("rows", 1)
    if rows > 1:
        r.capture_batch_graphs(rows)
    prompts = _prompts(case, seed)
    state = _State(case=case, runner=r, prompts=prompts, options=SamplingOptions(seed=seed), sids=[])
    if case["kind"] == "reply" or (case["kind"] == "batch" and case["model"] not in STACKS):
        for p in prompts:                               # the conversation so far
            sid = r.new_sequence()
            r.prefill(sid, p, want_logits=False)
            state["sids"].append(sid)
    if rows > 1:
        state["ring"] = [torch.zeros(rows, dtype=torch.int32).pin_memory() for _ in range(4)]
    return state


def run(state: dict):
    case = state["case"]
    if case["kind"] == "image":
        return state["encoder"].encode_pixels(state["pixels"])
    if case["kind"] == "batch":
        return _run_batch(state)
    r, p = state["runner"], state["prompts"][0]
    sid = state["sids"][0] if state["sids"] else r.new_sequence()
    tokens = list(r.generate(sid, p, state["options"], max_tokens=case["tokens"]))
    if not state["sids"]:
        r.free_sequence(sid)
    return dict(tokens=np.array(tokens), logits=r.logits[:1])


def _run_batch(state: dict):
    """Several requests admitted together and decoded in shared steps, two of them in flight."""
    r, prompts, o, case = state["runner"], state["prompts"], state["options"], state["case"]
    fresh = not state["sids"]
    sids = [r.new_sequence() for _ in prompts] if fresh else state["sids"]
    keep = [0 if fresh else len(p) - 1 for p in prompts]
    first = r.admit_many([(s, k, p[k:], o, p, o.seed + i) for i, (s, k, p) in enumerate(zip(sids, keep, prompts))])
    r.recompose([(o, p + [t], o.seed + i, 1) for i, (p, t) in enumerate(zip(prompts, first))], first)
    B, out, flight = len(prompts), [first], []
    for step in range(case["tokens"] - 1):
        r.decode_batch(sids, [len(p) + step for p in prompts])
        buf = state["ring"][step % 4]
        buf.copy_(r.s_out[:B], non_blocking=True)
        ev = torch.cuda.Event()
        ev.record()
        flight.append((buf, ev))
        if len(flight) == 2:
            _take(flight, out)
    while flight:
        _take(flight, out)
    logits = r.logits[:B].clone() if fresh else r.logits[:B]
    if fresh:
        for s in sids:
            r.free_sequence(s)
    return dict(tokens=np.array(out), logits=logits)


def _take(flight: list, out: list) -> None:
    buf, ev = flight.pop(0)
    ev.synchronize()
    out.append(buf.tolist())


def exact(case: dict, seed: int):
    if case["kind"] == "image":
        return _clip_exact(case, seed)
    forward = _stack_exact if case["model"] in STACKS else _gguf_exact
    logits = []
    for p, reply in zip(_prompts(case, seed), _replies(case, seed)):
        logits.append(forward(case, seed, p + reply[:-1]))      # the last token's logits come from the one before it
    return dict(tokens=None, logits=torch.cat(logits))


def _weight_bytes(case: dict) -> tuple[float, float, float]:
    """(bytes that one row's step reads, bytes in all, weights that one row multiplies)."""
    if case["kind"] == "image":
        n = case["layers"] * (4 * CLIP["E"] ** 2 + 2 * CLIP["E"] * CLIP["F"]) + CLIP["out"] * (CLIP["E"] + CLIP["out"])
        return 2.0 * n, 2.0 * n, float(n)
    if case["model"] in STACKS:
        E, pattern, H, G, D, F, X, top, Fs, (rh, rd, rv) = STACKS[case["model"]]
        w = 2.0 if case["ftype"] == "bf16" else 4.0
        mix = sum(E * (2 * H * D + 2 * G * D) if c == "a" else E * rh * (2 * rd + 3 * rv) for c in pattern)
        act = mix + len(pattern) * 3 * E * (top * F + Fs) + VOCAB * E
        return w * act, w * (act + len(pattern) * 3 * E * F * (X - top) + VOCAB * E), float(act)
    step = total = act = 0.0
    d = _dims(case)
    for name, (kind, rows, K, _s) in _Gguf(case, 0).mats.items():
        n = rows * K / BLOCK[kind][0] * BLOCK[kind][1]
        total += n
        if name != "token_embd":
            share = d["top"] / d["X"] if name.endswith("_exps") else 1.0
            step, act = step + n * share, act + rows * K * share
    return step, total, act


def work(case: dict) -> dict:
    one, total, act = _weight_bytes(case)
    if case["kind"] == "image":
        n = (case["size"] // CLIP["patch"]) ** 2 + 1
        return dict(bytes=total + 4.0 * n * CLIP["out"] + 12.0 * case["size"] ** 2,
                    flops=2.0 * n * act + 4.0 * case["layers"] * n * n * CLIP["E"])
    stack = case["model"] in STACKS
    if stack:
        E, pattern, H, G, D = STACKS[case["model"]][:5]
        layers, kv, qd = pattern.count("a"), (4.0 if case["ftype"] == "bf16" else 8.0) * G * D, H * D
        head, X, top = VOCAB * E * (2.0 if case["ftype"] == "bf16" else 4.0), STACKS[case["model"]][6], STACKS[case["model"]][7]
        all_w = total - head            # without the embedding, of which rows are read
    else:
        d = _dims(case)
        layers, kv, qd, X, top = d["L"], 4.0 * d["G"] * d["D"], d["E"], d["X"], d["top"]
        kind, rows, K, _s = _Gguf(case, 0).mats["token_embd"]
        all_w = total - rows * K / BLOCK[kind][0] * BLOCK[kind][1]
        head = VOCAB * d["E"]
    bytes_, flops = 0.0, 0.0
    rows = case.get("rows", 1)
    lengths = [case["prompt"] if rows == 1 else max(2, case["prompt"] * (2 + r % 3) // 3) for r in range(rows)]

    def step(n_each, starts):
        """One forward: n_each new rows per sequence after `starts` cached ones; all weights that any row needs once."""
        nonlocal bytes_, flops
        n = sum(n_each)
        share = 1.0 - (1.0 - top / X) ** n if X else 1.0
        bytes_ += one + (all_w - one) * max(0.0, (share - top / X) / (1.0 - top / X)) if X else all_w
        for a, s in zip(n_each, starts):
            bytes_ += layers * kv * (s + a)
            flops += 4.0 * layers * qd * a * (s + 0.5 * a)
        flops += 2.0 * act * n - 2.0 * VOCAB * (STACKS[case["model"]][0] if stack else SHAPES[case["model"]][0]) * (n - len(n_each))

    fresh = case["kind"] == "prompt" or stack
    step([n if fresh else 1 for n in lengths], [0 if fresh else n - 1 for n in lengths])
    for t in range(case["tokens"] - 1):
        step([1] * rows, [n + t for n in lengths])
    return dict(bytes=bytes_, flops=flops)


def tolerance(case: dict):
    """Relative errors of the logits or embedding rows against other implementations at the engine's precision: about four
    times the distance from the 64-bit results (image 5.5e-4, float32 3e-7, bfloat16 2.8e-3, quantised models with 8-bit
    activations 5.5e-3 at 8 layers and 9.5e-3 at 32)."""
    if case["kind"] == "image":
        return {"rel": 2.5e-3, "max": 0.03}
    if case["ftype"] == "f32":
        return {"rel": 5e-6, "max": 5e-5, "differ": 0.0}
    if case["ftype"] == "bf16":
        return {"rel": 1.2e-2, "max": 0.12, "differ": 0.0}
    return {"rel": 3e-2 if case["layers"] > 8 else 2e-2, "max": 0.2, "differ": 0.0}
