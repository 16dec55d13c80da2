"""The work that a user of the library has it do, as cases that can be timed and compared: single products over packed
weights, mixture-of-experts layers, latent attention, a whole decoder over GGUF blocks and one over plain bf16 rows, each
at its smallest, an ordinary and a large size, for one row and for many.

Sizes are those of the benchmark (`bench.py`): the Llama-3-8B and Qwen3-8B projections, the Qwen3-30B-A3B and DeepSeek-V3
expert layers, the DeepSeek-V3 attention block, four decoder layers of Qwen3-8B's sizes with a vocabulary of 32000, and
an attention and a scan layer of the benchmark's layered decoder.  Weights are normal, quantized here to real blocks.
"""
from __future__ import annotations

import json
import math
import os
import struct
import tempfile

import numpy as np
import torch

from joshua_amd import capi

DEV = "cuda"
f64 = torch.float64
TYPES = {"q4_k": (capi.Q4_K, 256, 144), "q6_k": (capi.Q6_K, 256, 210), "q8_0": (capi.Q8_0, 32, 34), "mxfp4": (capi.MXFP4, 32, 17)}

MOE = {  # type: hidden, inter, experts, used, sigmoid gates, groups, groups taken, factor on the weights, a shared expert
    "q4_k": dict(hidden=2048, inter=768, experts=128, used=8, sigmoid=False, groups=1, top_groups=1, scale=0.0, shared=False),
    "mxfp4": dict(hidden=7168, inter=2048, experts=256, used=8, sigmoid=True, groups=8, top_groups=4, scale=2.5, shared=True),
}
MLA = dict(n_embd=7168, n_head=128, q_lora_rank=1536, kv_lora_rank=512, qk_nope_head_dim=128, qk_rope_head_dim=64, v_head_dim=128,
           rms_eps=1e-6, rope_theta=10000.0, yarn_factor=40.0, yarn_mscale_all_dim=1.0, yarn_orig_context_length=4096)
QWEN3 = dict(n_layer=4, hidden=4096, n_head=32, n_kv_head=8, head_dim=128, ffn=12288, vocab=32000, rms_eps=1e-6, rope_theta=1e6)
BOZOSUN = {
    "architecture": "Bozosun", "vocab": 32000, "width": 4096, "embedding": {"scale": 8.0}, "norm": {"eps": 1e-6}, "residual_mult": 0.5,
    "layers": [
        {"type": "attention", "mixer": {"heads": 32, "kv_heads": 8, "dim": 128, "vdim": 128, "scale": 128 ** -0.5, "v_mix": False,
                                        "rot": {"dims": 128, "base": 1e6, "scaling": {"factor": 4.0, "original": 8192, "fast": 32.0, "slow": 1.0}}},
         "mlp": {"kind": "dense", "ff": 12288, "limit": 7.0}},
        {"type": "mamba1", "mixer": {"inner": 8192, "state": 16, "dt_rank": 256, "conv": 4}, "mlp": {"kind": "dense", "ff": 12288, "limit": 7.0}},
    ],
}


def listed():
    return [
        # one row through the smallest projection of a decode step: latency
        dict(name="row_q8_0", path="matmul", type="q8_0", m=1, n=4096, k=4096),
        # one row through a feed-forward projection: the benchmark's headline, bound by the weights' bytes
        dict(name="row_q4_k", path="matmul", type="q4_k", m=1, n=14336, k=4096),
        # a batch of decoding sequences, or a speculative step, through the same projection
        dict(name="batch_q4_k", path="matmul", type="q4_k", m=16, n=14336, k=4096),
        # a prompt's feed-forward projection
        dict(name="prompt_q4_k", path="matmul", type="q4_k", m=512, n=14336, k=4096),
        # a prompt of any length through a down projection, in the type that a Q4_K_M file keeps for it
        dict(name="ragged_q6_k", path="matmul", type="q6_k", m=333, n=4096, k=12288),
        # a prompt through a Qwen3-30B-A3B expert layer: 32 rows an expert
        dict(name="experts_prompt", path="moe", type="q4_k", tokens=512),
        # a batch of decoding sequences through a DeepSeek-V3 expert layer, nearly every expert for a row or two
        dict(name="experts_batch", path="moe", type="mxfp4", tokens=64),
        # latent attention of DeepSeek-V3: a long prompt in chunks, and single tokens behind a short one
        dict(name="latent_prompt", path="mla", tokens=4096, chunk=512, steps=0),
        dict(name="latent_steps", path="mla", tokens=61, chunk=61, steps=48),
        # a decoder of Qwen3-8B's sizes: a long prompt; an ordinary prompt and the tokens that follow
        dict(name="decoder_prompt", path="decoder", prompt=2048, steps=0),
        dict(name="decoder_steps", path="decoder", prompt=200, steps=32),
        # a decoder with plain bf16 weights from a folder: a prompt and the first tokens behind it
        dict(name="folder_turn", path="folder", prompt=512, steps=8),
    ]


def draw(rng):
    def log(lo, hi):
        return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))

    path = rng.choice(["matmul"] * 4 + ["moe", "mla", "decoder", "folder"])
    if path == "matmul":
        return dict(path=path, type=rng.choice(sorted(TYPES)), m=log(1, 512), n=log(1024, 14336), k=256 * rng.randint(8, 48))
    if path == "moe":
        return dict(path=path, type=rng.choice(sorted(MOE)), tokens=log(1, 512))
    if path == "mla":
        return dict(path=path, tokens=log(1, 3000), chunk=rng.randint(100, 512), steps=rng.randint(0, 48))
    return dict(path=path, prompt=log(1, 2000), steps=rng.randint(0, 24 if path == "decoder" else 12))


# ---- weights: normal values as packed blocks ---------------------------------------------------------------------

def _f16(x):
    """Scales as the block holds them: (bytes [.., 2], the value in f32)."""
    h = x.to(torch.float16)
    return h.unsqueeze(-1).view(torch.uint8), h.float()


def _pack(kind, w):
    """[n] normal values -> packed bytes."""
    if kind == "q8_0":
        x = w.view(-1, 32)
        db, d = _f16(x.abs().amax(1) / 127)
        q = torch.round(x / d[:, None]).clamp(-127, 127).to(torch.int8).view(torch.uint8)
        return torch.cat([db, q], 1)
    if kind == "mxfp4":
        x = w.view(-1, 32)
        e = torch.floor(torch.log2(x.abs().amax(1).clamp_min(1e-20))) - 2
        x = x * torch.exp2(-e)[:, None]
        q = torch.bucketize(x.abs(), torch.tensor([0.25, 0.75, 1.25, 1.75, 2.5, 3.5, 5.0], device=w.device), out_int32=True).to(torch.uint8)
        q |= (x < 0).to(torch.uint8) << 3
        return torch.cat([(e + 127).to(torch.uint8)[:, None], q[:, :16] | q[:, 16:] << 4], 1)
    if kind == "q6_k":
        x = w.view(-1, 16, 16)
        s = x.abs().amax(2) / 31
        db, d = _f16(s.amax(1) / 127)
        sc = torch.round(s / d[:, None]).clamp(1, 127)
        q = (torch.round(x / (d[:, None] * sc)[..., None]).clamp(-32, 31) + 32).to(torch.uint8).view(-1, 2, 4, 32)
        ql = (q[:, :, :2] & 15) | (q[:, :, 2:] & 15) << 4
        qh = q[:, :, 0] >> 4 | q[:, :, 1] >> 4 << 2 | q[:, :, 2] >> 4 << 4 | q[:, :, 3] >> 4 << 6
        return torch.cat([ql.reshape(-1, 128), qh.reshape(-1, 64), sc.to(torch.uint8), db], 1)
    x = w.view(-1, 8, 32)
    lo = x.amin(2).clamp_max(0)
    db, d = _f16((x.amax(2) - lo).amax(1) / (15 * 63))
    mb, dmin = _f16((-lo).amax(1) / 63)
    sc = torch.round((x.amax(2) - lo) / (15 * d[:, None])).clamp(1, 63)
    mn = torch.round(-lo / dmin[:, None]).clamp(0, 63)
    q = torch.round((x + (dmin[:, None] * mn)[..., None]) / (d[:, None] * sc)[..., None]).clamp(0, 15).to(torch.uint8).view(-1, 4, 2, 32)
    sc, mn = sc.to(torch.uint8), mn.to(torch.uint8)
    low, high = slice(0, 4), slice(4, 8)
    six = torch.cat([sc[:, low] | sc[:, high] >> 4 << 6, mn[:, low] | mn[:, high] >> 4 << 6, (sc[:, high] & 15) | (mn[:, high] & 15) << 4], 1)
    return torch.cat([db, mb, six, (q[:, :, 0] | q[:, :, 1] << 4).reshape(-1, 128)], 1)


def _values(kind, b):
    """Packed bytes -> the values they stand for, in 64 bits."""
    _, elems, size = TYPES[kind]
    b = b.view(-1, size)

    def scale(at):
        return b[:, at:at + 2].contiguous().view(torch.float16).to(f64)

    if kind == "q8_0":
        return (scale(0) * b[:, 2:].contiguous().view(torch.int8).to(f64)).view(-1)
    if kind == "mxfp4":
        e2m1 = torch.tensor([0, 0.5, 1, 1.5, 2, 3, 4, 6, 0, -0.5, -1, -1.5, -2, -3, -4, -6], dtype=f64, device=b.device)
        return (e2m1[torch.cat([b[:, 1:] & 15, b[:, 1:] >> 4], 1).int()] * torch.exp2(b[:, :1].to(f64) - 127)).view(-1)
    if kind == "q6_k":
        ql, qh = b[:, :128].reshape(-1, 2, 2, 32), b[:, 128:192].reshape(-1, 2, 32)
        q = torch.cat([ql & 15, ql >> 4], 2) | torch.stack([(qh >> 2 * t & 3) << 4 for t in range(4)], 2)
        sc = b[:, 192:208].contiguous().view(torch.int8).to(f64) * scale(208)
        return ((q.to(f64) - 32).view(-1, 16, 16) * sc[..., None]).view(-1)
    s, q = b[:, 4:16], b[:, 16:].reshape(-1, 4, 1, 32)
    sc = torch.cat([s[:, :4] & 63, (s[:, 8:] & 15) | s[:, :4] >> 6 << 4], 1).to(f64) * scale(0)
    mn = torch.cat([s[:, 4:8] & 63, s[:, 8:] >> 4 | s[:, 4:8] >> 6 << 4], 1).to(f64) * scale(2)
    return (torch.cat([q & 15, q >> 4], 2).reshape(-1, 8, 32).to(f64) * sc[..., None] - mn[..., None]).view(-1)


class Source:
    """Seeded inputs, made on the device in the order in which they are asked for."""

    def __init__(self, seed):
        self.g = torch.Generator(device=DEV).manual_seed(int(seed) * 7919 + 11)

    def normal(self, *shape, sigma=1.0, mean=0.0):
        return torch.randn(*shape, generator=self.g, device=DEV) * sigma + mean

    def ids(self, n, bound):
        return torch.randint(0, bound, (n,), generator=self.g, device=DEV).cpu().numpy().astype(np.uint32)

    def blocks(self, kind, n, k, sigma):
        """An n x k matrix as packed blocks."""
        _, elems, size = TYPES[kind]
        out = torch.empty(n * k // elems, size, dtype=torch.uint8, device=DEV)
        step = 1 << 26
        for at in range(0, n * k, step):
            most = min(step, n * k - at)
            out[at // elems:(at + most) // elems] = _pack(kind, self.normal(most, sigma=sigma))
        return out.view(-1)


def _weight(kind, blocks, n, k):
    torch.cuda.synchronize()
    return capi.Weight.upload_device(TYPES[kind][0], blocks.data_ptr(), blocks.numel(), n, k)


def _stream():
    return torch.cuda.current_stream().cuda_stream


# ---- one product -------------------------------------------------------------------------------------------------------

def _matmul_inputs(c, seed):
    s = Source(seed)
    return s.blocks(c["type"], c["n"], c["k"], 0.02), s.normal(c["m"], c["k"])


def _matmul_prepare(c, seed):
    blocks, x = _matmul_inputs(c, seed)
    return dict(m=c["m"], w=_weight(c["type"], blocks, c["n"], c["k"]), x=x, y=torch.zeros(c["m"], c["n"], device=DEV))


def _matmul_run(s):
    x, y = s["x"], s["y"]
    s["w"].matmul_t_dev(s["m"], x.data_ptr(), x.numel(), y.data_ptr(), y.numel(), _stream())
    return y


def _matmul_exact(c, seed):
    blocks, x = _matmul_inputs(c, seed)
    return x.to(f64) @ _values(c["type"], blocks).view(c["n"], c["k"]).T


# ---- a mixture-of-experts layer ------------------------------------------------------------------------------------------

def _moe_inputs(c, seed):
    p, s = MOE[c["type"]], Source(seed)
    E, h, f = p["experts"], p["hidden"], p["inter"]
    yield "router", s.normal(E, h, sigma=0.02)
    yield "bias", s.normal(E, sigma=0.01)
    yield "x", s.normal(c["tokens"], h)
    for name, n, k in (("gate", f, h), ("up", f, h), ("down", h, f)):
        if p["shared"]:
            yield "shared_" + name, s.blocks(c["type"], n, k, 0.02)
        yield name, s.blocks(c["type"], E * n, k, 0.02)


def _moe_prepare(c, seed):
    p, st = MOE[c["type"]], {}
    E, h, f = p["experts"], p["hidden"], p["inter"]
    for name, t in _moe_inputs(c, seed):  # one stack of experts at a time as torch memory
        role = name.split("_")[-1]
        if role in ("gate", "up", "down"):
            n, k = (h, f) if role == "down" else (f, h)
            t = _weight(c["type"], t, n if "shared" in name else E * n, k)
        st[name] = t
    cfg = capi.MoeConfig(E, p["used"], h, f, int(p["sigmoid"]), 1, p["scale"], p["groups"], p["top_groups"])
    shared = tuple(st["shared_" + r] for r in ("gate", "up", "down")) if p["shared"] else None
    moe = capi.Moe(cfg, st["router"].cpu().numpy(), st["gate"], st["up"], st["down"],
                   router_bias=st["bias"].cpu().numpy() if p["sigmoid"] else None, shared=shared)
    return dict(moe=moe, x=st["x"], y=torch.zeros_like(st["x"]), tokens=c["tokens"])


def _moe_run(s):
    s["moe"].forward_dev(s["tokens"], s["x"].data_ptr(), s["y"].data_ptr(), _stream())
    return s["y"]


def _moe_exact(c, seed):
    p = MOE[c["type"]]
    E, h, f = p["experts"], p["hidden"], p["inter"]
    st = dict(_moe_inputs(c, seed))
    x, T = st["x"].to(f64), c["tokens"]
    logits = x @ st["router"].to(f64).T
    probs = torch.sigmoid(logits) if p["sigmoid"] else torch.softmax(logits, 1)
    chosen = probs + st["bias"].to(f64) if p["sigmoid"] else probs
    if p["groups"] > 1:
        by_group = chosen.view(T, p["groups"], -1)
        best = by_group.topk(2, 2)[0].sum(2).topk(p["top_groups"], 1)[1]
        mask = torch.zeros(T, p["groups"], dtype=torch.bool, device=DEV).scatter_(1, best, True)
        chosen = by_group.masked_fill(~mask[..., None], -1e30).reshape(T, E)
    ids = chosen.topk(p["used"], 1)[1]
    wt = probs.gather(1, ids)
    wt = wt / wt.sum(1, keepdim=True) * (p["scale"] or 1.0)

    def mlp(x, blocks):
        g, u, d = (_values(c["type"], b).view(n, k) for b, n, k in zip(blocks, (f, f, h), (h, h, f)))
        return (torch.nn.functional.silu(x @ g.T) * (x @ u.T)) @ d.T

    y = mlp(x, [st["shared_" + r] for r in ("gate", "up", "down")]) if p["shared"] else torch.zeros_like(x)
    stacks = [st[r].view(E, -1) for r in ("gate", "up", "down")]
    for e in torch.unique(ids).tolist():
        t, slot = torch.nonzero(ids == e, as_tuple=True)
        y.index_add_(0, t, mlp(x[t], [s[e] for s in stacks]) * wt[t, slot][:, None])
    return y


# ---- rotary positions ---------------------------------------------------------------------------------------------------

def _yarn(dims, base, factor, original, fast, slow):
    """(frequency of each pair, factor on cosine and sine)."""
    i = torch.arange(dims // 2, dtype=f64, device=DEV)
    f = base ** (-2 * i / dims)

    def turns(t):
        return dims * math.log(original / (2 * math.pi * t)) / (2 * math.log(base))

    lo, hi = max(math.floor(turns(fast)), 0), min(math.ceil(turns(slow)), dims - 1)
    ramp = ((i - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return f / factor * ramp + f * (1 - ramp), 0.1 * math.log(factor) + 1


def _rotate(v, freq, mag, interleaved):
    """v [T, heads, d]: pairs of neighbours, or of one half with the other, turn with the position."""
    a = torch.arange(v.shape[0], dtype=f64, device=DEV)[:, None, None] * freq
    c, s = mag * torch.cos(a), mag * torch.sin(a)
    x, y = (v[..., 0::2], v[..., 1::2]) if interleaved else v.chunk(2, -1)
    x, y = x * c - y * s, y * c + x * s
    return torch.stack([x, y], -1).flatten(-2) if interleaved else torch.cat([x, y], -1)


def _attend(q, k, v, scale):
    """Causal softmax attention; q [T, heads, d], k and v [T, their heads, d]."""
    T, heads, _ = q.shape
    out, rep = torch.empty(T, heads, v.shape[2], dtype=f64, device=DEV), heads // k.shape[1]
    hidden = torch.ones(T, T, dtype=torch.bool, device=DEV).triu(1)
    for h in range(heads):
        s = (q[:, h] @ k[:, h // rep].T * scale).masked_fill(hidden, -math.inf)
        out[:, h] = torch.softmax(s, 1) @ v[:, h // rep]
    return out.view(T, -1)


def _rms(x, w, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps) * w


# ---- latent attention -----------------------------------------------------------------------------------------------------

def _mla_shapes():
    m = MLA
    H, nope, rope, R = m["n_head"], m["qk_nope_head_dim"], m["qk_rope_head_dim"], m["kv_lora_rank"]
    return {"q_a": (m["q_lora_rank"], m["n_embd"]), "q_b": (H * (nope + rope), m["q_lora_rank"]), "kv_a": (R + rope, m["n_embd"]),
            "kv_b": (H * (nope + m["v_head_dim"]), R), "o": (m["n_embd"], H * m["v_head_dim"])}


def _mla_inputs(c, seed):
    s = Source(seed)
    st = {name: s.blocks("q4_k", n, k, 0.02) for name, (n, k) in _mla_shapes().items()}
    st["q_norm"], st["kv_norm"] = s.normal(MLA["q_lora_rank"], sigma=0.1, mean=1.0), s.normal(MLA["kv_lora_rank"], sigma=0.1, mean=1.0)
    st["x"] = s.normal(c["tokens"] + c["steps"], MLA["n_embd"])
    return st


def _mla_prepare(c, seed):
    st = _mla_inputs(c, seed)
    w = {name: _weight("q4_k", st[name], n, k) for name, (n, k) in _mla_shapes().items()}
    cfg = capi.MlaConfig(n_ctx=c["tokens"] + c["steps"], **MLA)
    mla = capi.Mla(cfg, (w["q_a"], st["q_norm"].cpu().numpy(), w["q_b"]), w["kv_a"], st["kv_norm"].cpu().numpy(), w["kv_b"], w["o"])
    return dict(mla=mla, case=dict(c), x=st["x"], y=torch.zeros_like(st["x"]))


def _mla_run(s):
    c, x, y, row = s["case"], s["x"], s["y"], 4 * MLA["n_embd"]
    s["mla"].reset()
    pos, end = 0, c["tokens"] + c["steps"]
    while pos < end:
        n = min(c["chunk"], c["tokens"] - pos) if pos < c["tokens"] else 1
        s["mla"].forward_dev(n, pos, x.data_ptr() + row * pos, y.data_ptr() + row * pos, _stream())
        pos += n
    return y


def _mla_exact(c, seed):
    st, m = _mla_inputs(c, seed), MLA
    H, nope, rope, R, eps = m["n_head"], m["qk_nope_head_dim"], m["qk_rope_head_dim"], m["kv_lora_rank"], m["rms_eps"]
    w = {name: _values("q4_k", st[name]).view(n, k) for name, (n, k) in _mla_shapes().items()}
    x = st["x"].to(f64)
    T = len(x)
    freq, mag = _yarn(rope, m["rope_theta"], m["yarn_factor"], m["yarn_orig_context_length"], 32.0, 1.0)
    q = (_rms(x @ w["q_a"].T, st["q_norm"].to(f64), eps) @ w["q_b"].T).view(T, H, nope + rope)
    kv = x @ w["kv_a"].T
    up = (_rms(kv[:, :R], st["kv_norm"].to(f64), eps) @ w["kv_b"].T).view(T, H, -1)
    q = torch.cat([q[..., :nope], _rotate(q[..., nope:], freq, mag, True)], -1)
    k = torch.cat([up[..., :nope], _rotate(kv[:, None, R:], freq, mag, True).expand(T, H, rope)], -1)
    return _attend(q, k, up[..., nope:], mag * mag / math.sqrt(nope + rope)) @ w["o"].T


# ---- a decoder over GGUF blocks ---------------------------------------------------------------------------------------------

def _decoder_inputs(c, seed):
    """(tensor name, type or f32, rows, values), then the tokens.  The types are those of a Q4_K_M file."""
    m, s = QWEN3, Source(seed)
    h, d, f = m["hidden"], m["head_dim"], m["ffn"]
    plan = [("token_embd", "q4_k", m["vocab"], h), ("output_norm", "f32", h, 0), ("output", "q6_k", m["vocab"], h)]
    for i in range(m["n_layer"]):
        more = "q6_k" if i >= 2 else "q4_k"
        p = f"blk.{i}."
        plan += [(p + "attn_norm", "f32", h, 0), (p + "attn_q", "q4_k", m["n_head"] * d, h), (p + "attn_k", "q4_k", m["n_kv_head"] * d, h),
                 (p + "attn_v", "q8_0" if i == 3 else more, m["n_kv_head"] * d, h), (p + "attn_q_norm", "f32", d, 0),
                 (p + "attn_k_norm", "f32", d, 0), (p + "attn_output", "q4_k", h, m["n_head"] * d), (p + "ffn_norm", "f32", h, 0),
                 (p + "ffn_gate", "q4_k", f, h), (p + "ffn_up", "q4_k", f, h), (p + "ffn_down", more, h, f)]
    for name, kind, n, k in plan:
        yield name, kind, n, s.normal(n, sigma=0.1, mean=1.0) if kind == "f32" else s.blocks(kind, n, k, k ** -0.5)
    yield "tokens", "", 0, s.ids(c["prompt"] + c["steps"], m["vocab"])


def _decoder_prepare(c, seed):
    m = QWEN3
    model = capi.Qwen3(capi.Qwen3Config(m["n_layer"], m["hidden"], m["n_head"], m["n_kv_head"], m["head_dim"], m["ffn"], m["vocab"],
                                        c["prompt"] + c["steps"], m["rms_eps"], m["rope_theta"]))
    for name, kind, _, t in _decoder_inputs(c, seed):
        if name == "tokens":
            return dict(model=model, prompt=c["prompt"], tokens=t)
        model.set_tensor(name + ".weight", 0 if kind == "f32" else TYPES[kind][0], t.cpu().numpy())


def _turn(s):
    """A new sequence: the prompt in one step, then known tokens one at a time; the logits of each step."""
    model, tokens, n = s["model"], s["tokens"], s["prompt"]
    model.reset()
    logits = [model.forward(tokens[:n], 0)]
    for pos in range(n, len(tokens)):
        logits.append(model.forward(tokens[pos:pos + 1], pos))
    return np.stack(logits)


def _decoder_exact(c, seed):
    m, w = QWEN3, {}
    for name, kind, n, t in _decoder_inputs(c, seed):
        w[name] = t if name == "tokens" else (kind, n, t)

    def mat(name):
        kind, n, t = w[name]
        return t.to(f64) if kind == "f32" else _values(kind, t).view(n, -1)

    H, G, d, eps = m["n_head"], m["n_kv_head"], m["head_dim"], m["rms_eps"]
    x = mat("token_embd")[torch.from_numpy(w["tokens"].astype(np.int64)).to(DEV)]
    T = len(x)
    freq = m["rope_theta"] ** (-torch.arange(0, d, 2, dtype=f64, device=DEV) / d)
    for i in range(m["n_layer"]):
        p = f"blk.{i}."
        a = _rms(x, mat(p + "attn_norm"), eps)
        q, k, v = ((a @ mat(p + "attn_" + r).T).view(T, -1, d) for r in "qkv")
        q, k = (_rotate(_rms(y, mat(p + "attn_" + r + "_norm"), eps), freq, 1.0, False) for y, r in ((q, "q"), (k, "k")))
        x = x + _attend(q, k, v, d ** -0.5) @ mat(p + "attn_output").T
        a = _rms(x, mat(p + "ffn_norm"), eps)
        x = x + (torch.nn.functional.silu(a @ mat(p + "ffn_gate").T) * (a @ mat(p + "ffn_up").T)) @ mat(p + "ffn_down").T
    return _rms(x[c["prompt"] - 1:], mat("output_norm"), eps) @ mat("output").T


# ---- a decoder with plain rows ---------------------------------------------------------------------------------------------

def _folder_inputs(c, seed):
    """name -> bf16 values, and the tokens."""
    g, s = BOZOSUN, Source(seed)
    w = g["width"]

    def matrix(n, k):
        return s.normal(n, k, sigma=k ** -0.5)

    def norm(name):
        return {name: s.normal(w, sigma=0.2, mean=1.0), name + ".b": s.normal(w, sigma=0.1)}

    t = {"embed": s.normal(g["vocab"], w)}
    for i, layer in enumerate(g["layers"]):
        p, m, ff = f"l{i}.", layer["mixer"], layer["mlp"]["ff"]
        for name in ("norm1", "norm1b", "norm2", "norm2b"):
            t.update(norm(p + name))
        x = p + "mix."
        if layer["type"] == "attention":
            t.update({x + "q": matrix(m["heads"] * m["dim"], w), x + "k": matrix(m["kv_heads"] * m["dim"], w),
                      x + "v": matrix(m["kv_heads"] * m["vdim"], w), x + "o": matrix(w, m["heads"] * m["vdim"])})
        else:
            C, N, R = m["inner"], m["state"], m["dt_rank"]
            slow = 0.7 * torch.log(1.0 + torch.arange(N, device=DEV)) - 1.0
            t.update({x + "in": matrix(2 * C, w), x + "conv": s.normal(C, m["conv"], sigma=0.6), x + "conv.b": s.normal(C, sigma=0.3),
                      x + "x": matrix(R + 2 * N, C), x + "dt": matrix(C, R), x + "dt.b": s.normal(C, mean=-2.0),
                      x + "A_log": s.normal(C, N, sigma=0.3) + slow, x + "D": s.normal(C, sigma=0.6), x + "o": matrix(w, C)})
        t.update({p + "mlp.gate": matrix(ff, w), p + "mlp.up": matrix(ff, w), p + "mlp.down": matrix(w, ff)})
    t.update(norm("final.norm"))
    t["head"] = matrix(g["vocab"], w)
    return {name: v.to(torch.bfloat16) for name, v in t.items()}, s.ids(c["prompt"] + c["steps"], g["vocab"])


def _folder_prepare(c, seed):
    tensors, tokens = _folder_inputs(c, seed)
    header, at = {}, 0
    for name, t in tensors.items():
        header[name] = {"dtype": "BF16", "shape": list(t.shape), "data_offsets": [at, at + 2 * t.numel()]}
        at += 2 * t.numel()
    text = json.dumps(header).encode()
    with tempfile.TemporaryDirectory() as folder:
        with open(os.path.join(folder, "config.json"), "w") as f:
            json.dump(BOZOSUN, f)
        with open(os.path.join(folder, "model.safetensors"), "wb") as f:
            f.write(struct.pack("<Q", len(text)) + text)
            for t in tensors.values():
                f.write(t.view(torch.uint8).cpu().numpy().data)
        model = capi.Model(folder, n_ctx=c["prompt"] + c["steps"])
    return dict(model=model, prompt=c["prompt"], tokens=tokens)


def _folder_exact(c, seed):
    tensors, tokens = _folder_inputs(c, seed)
    g, eps, mult = BOZOSUN, BOZOSUN["norm"]["eps"], BOZOSUN["residual_mult"]

    def mat(name):
        return tensors[name].to(f64)

    def norm(x, name):
        return torch.nn.functional.layer_norm(x, x.shape[-1:], mat(name), mat(name + ".b"), eps)

    def attention(h, p, m):
        T, rot = len(h), m["rot"]
        q, k, v = ((h @ mat(p + r).T).view(T, -1, d) for r, d in (("q", m["dim"]), ("k", m["dim"]), ("v", m["vdim"])))
        freq, mag = _yarn(rot["dims"], rot["base"], **rot["scaling"])
        q, k = (_rotate(y, freq, mag, True) for y in (q, k))
        return _attend(q, k, v, m["scale"])

    def scan(h, p, m):
        C, N, R, taps = m["inner"], m["state"], m["dt_rank"], m["conv"]
        x, z = (h @ mat(p + "in").T).split(C, 1)
        full = torch.cat([torch.zeros(taps - 1, C, dtype=f64, device=DEV), x])
        x = torch.nn.functional.silu(sum(full[j:j + len(x)] * mat(p + "conv")[:, j] for j in range(taps)) + mat(p + "conv.b"))
        dt, B, Q = (x @ mat(p + "x").T).split([R, N, N], 1)
        dt = dt @ mat(p + "dt").T + mat(p + "dt.b")
        dt = torch.logaddexp(dt, torch.zeros_like(dt))
        A, S, y = -torch.exp(mat(p + "A_log")), torch.zeros(C, N, dtype=f64, device=DEV), []
        for t in range(len(x)):
            S = torch.exp(dt[t][:, None] * A) * S + (dt[t] * x[t])[:, None] * B[t]
            y.append(S @ Q[t])
        return (torch.stack(y) + mat(p + "D") * x) * torch.nn.functional.silu(z)

    x = mat("embed")[torch.from_numpy(tokens.astype(np.int64)).to(DEV)] * g["embedding"]["scale"]
    for i, layer in enumerate(g["layers"]):
        p = f"l{i}."
        y = (attention if layer["type"] == "attention" else scan)(norm(x, p + "norm1"), p + "mix.", layer["mixer"])
        x = x + mult * norm(y @ mat(p + "mix.o").T, p + "norm1b")
        h, limit = norm(x, p + "norm2"), layer["mlp"]["limit"]
        a, u = (h @ mat(p + "mlp.gate").T).clamp(max=limit), (h @ mat(p + "mlp.up").T).clamp(-limit, limit)
        x = x + mult * norm((a * torch.sigmoid(1.702 * a) * (u + 1)) @ mat(p + "mlp.down").T, p + "norm2b")
    return norm(x[c["prompt"] - 1:], "final.norm") @ mat("head").T


# ---- what a measurement calls ----------------------------------------------------------------------------------------------

_PREPARE = dict(matmul=_matmul_prepare, moe=_moe_prepare, mla=_mla_prepare, decoder=_decoder_prepare, folder=_folder_prepare)
_RUN = dict(matmul=_matmul_run, moe=_moe_run, mla=_mla_run, decoder=_turn, folder=_turn)
_EXACT = dict(matmul=_matmul_exact, moe=_moe_exact, mla=_mla_exact, decoder=_decoder_exact, folder=_folder_exact)


def prepare(case, seed):
    return dict(_PREPARE[case["path"]](case, seed), path=case["path"])


def run(state):
    return _RUN[state["path"]](state)


def exact(case, seed):
    return _EXACT[case["path"]](case, seed)


def _causal(first, n):
    """Pairs of a token and one that it sees, for n tokens behind `first`."""
    return n * first + n * (n + 1) // 2


def work(case):
    """Packed weights once a step (a call to the library), inputs and results once; two operations a weight and row, and
    a pair of tokens' scores and sums in attention."""
    c = case
    if c["path"] == "matmul":
        _, elems, size = TYPES[c["type"]]
        m, n, k = c["m"], c["n"], c["k"]
        return dict(bytes=n * k // elems * size + 4 * m * (n + k), flops=2 * m * n * k)
    if c["path"] == "moe":
        p = MOE[c["type"]]
        _, elems, size = TYPES[c["type"]]
        E, h, f, T = p["experts"], p["hidden"], p["inter"], c["tokens"]
        met = E * (1 - (1 - p["used"] / E) ** T) + p["shared"]  # experts that some token chose, on average
        each = p["used"] + p["shared"]
        return dict(bytes=int(met * 3 * h * f // elems * size) + 4 * E * h + 8 * T * h, flops=6 * T * each * h * f + 2 * T * E * h)
    if c["path"] == "mla":
        m, T, steps = MLA, c["tokens"], c["steps"]
        calls = -(-T // c["chunk"]) + steps
        n = sum(a * b for a, b in _mla_shapes().values())
        seen = sum(min(T, i + c["chunk"]) for i in range(0, T, c["chunk"])) + sum(range(T + 1, T + steps + 1))
        head = m["qk_nope_head_dim"] + m["qk_rope_head_dim"] + m["v_head_dim"]
        return dict(bytes=calls * n // 256 * 144 + 4 * (m["kv_lora_rank"] + m["qk_rope_head_dim"]) * seen + 8 * (T + steps) * m["n_embd"],
                    flops=2 * (T + steps) * n + 2 * m["n_head"] * head * _causal(0, T + steps))
    T, steps = c["prompt"], c["steps"]
    if c["path"] == "decoder":
        m = QWEN3
        h, f, kv, q = m["hidden"], m["ffn"], m["n_kv_head"] * m["head_dim"], m["n_head"] * m["head_dim"]
        rest = h * (2 * q + kv) + 2 * h * f
        layers = 2 * (rest + h * kv + h * f) * 144 // 256 + 2 * rest * 144 // 256 + h * (kv + 2 * f) * 210 // 256 + h * kv * 34 // 32
        n, head, width = m["n_layer"] * (rest + h * (kv + f)), h * m["vocab"], 144 * h // 256
        cache, pair = m["n_layer"] * 8 * kv, m["n_layer"] * 4 * q
        return dict(bytes=(1 + steps) * (layers + head * 210 // 256 + 4 * m["vocab"]) + (T + steps) * width + cache * (T + _causal(T, steps)),
                    flops=2 * (T + steps) * n + 2 * (1 + steps) * head + pair * _causal(0, T + steps))
    g = BOZOSUN
    w, (a, b) = g["width"], (layer["mixer"] for layer in g["layers"])
    q, kv, C = a["heads"] * a["dim"], a["kv_heads"] * a["dim"], b["inner"]
    n = w * (2 * q + 2 * kv) + 6 * w * g["layers"][0]["mlp"]["ff"] + 3 * w * C + C * (2 * b["dt_rank"] + 2 * b["state"])
    head = w * g["vocab"]
    return dict(bytes=(1 + steps) * (2 * n + 2 * head + 4 * g["vocab"] + 8 * C * b["state"]) + 2 * (T + steps) * w + 4 * kv * (T + _causal(T, steps)),
                flops=2 * (T + steps) * (n + 4 * C * b["state"]) + 2 * (1 + steps) * head + 4 * q * _causal(0, T + steps))


def tolerance(case):
    """About four times what the library's results were seen to lie from `exact` (2.7e-5 in products over blocks with the
    activations in 16-bit fixed point, 7e-5 in expert layers, 1e-4 in latent attention, 1.6e-4 behind four decoder
    layers, 2.8e-4 behind two layers of bf16), or would with the f16 activations that some 17 to 63 rows go through."""
    return {"rel": {"matmul": 6e-4, "moe": 6e-4, "mla": 6e-4, "decoder": 8e-4, "folder": 2e-3}[case["path"]]}
