"""Multi-head latent attention on the GPU (absorbed form, latent cache) against the numpy
restatement of the reference's unabsorbed Attention::forward (oracle/mla.py), through the C ABI.
Bound: |gpu - ref| <= 1e-3 * max(|ref|, 1) on the block's output."""
import numpy as np
import pytest

import oracle
from oracle import mla as om
from joshua_amd import capi, synth
from joshua_amd.synth import normal

pytestmark = pytest.mark.gpu


def close(got, want, tol=1e-3):
    """Element by element, the bound of the other parity tests."""
    return bool(np.all(np.abs(got - want) <= tol * np.maximum(np.abs(want), 1.0)))


def quantized(qtype, seed, n, k, scale=1.0):
    """Random weights as blocks of `qtype` (n rows of k)."""
    w = (normal(seed, (n, k)) * np.float32(scale)).astype(np.float32)
    return synth.quantize(qtype, w)


def build(c, qtype=capi.Q8_0, seed=100, dense_kv_b=False):
    """Oracle tensors and the device object over the same blocks."""
    nh, lkv, npe, r, vh, h = c["n_head"], c["kv_lora_rank"], c["qk_nope"], c["qk_rope"], c["v_head_dim"], c["n_embd"]
    qd = npe + r
    shapes = {"kv_a_mqa": (lkv + r, h), "kv_b": (nh * (npe + vh), lkv), "o": (h, nh * vh)}
    if c["q_lora_rank"]:
        shapes.update(q_a=(c["q_lora_rank"], h), q_b=(nh * qd, c["q_lora_rank"]))
    else:
        shapes["q"] = (nh * qd, h)
    t, w = {}, {}
    for i, (name, (n, k)) in enumerate(sorted(shapes.items())):
        if name == "kv_b" and dense_kv_b:
            t[name] = (0, (normal(seed + i, (n, k)) / np.float32(np.sqrt(k))).astype(np.float32))
            continue
        blocks = quantized(qtype, seed + i, n, k, 1.0 / np.sqrt(k))
        t[name] = (qtype, blocks)
        w[name] = capi.Weight.upload(qtype, blocks, n, k)
    t["kv_a_norm"] = (1.0 + 0.1 * normal(seed + 20, (lkv,))).astype(np.float32)
    if c["q_lora_rank"]:
        t["q_a_norm"] = (1.0 + 0.1 * normal(seed + 21, (c["q_lora_rank"],))).astype(np.float32)
    y = c.get("yarn")
    cfg = capi.MlaConfig(n_embd=h, n_head=nh, q_lora_rank=c["q_lora_rank"], kv_lora_rank=lkv, qk_nope_head_dim=npe,
                         qk_rope_head_dim=r, v_head_dim=vh, n_ctx=c["context_length"], rms_eps=c["rms_eps"],
                         rope_theta=c["rope_theta"], yarn_factor=y["factor"] if y else 0.0,
                         yarn_mscale_all_dim=y["mscale_all_dim"] if y else 0.0,
                         yarn_orig_context_length=y["orig_context_length"] if y else 0)
    q = (w["q_a"], t["q_a_norm"], w["q_b"]) if c["q_lora_rank"] else w["q"]
    dev = capi.Mla(cfg, q, w["kv_a_mqa"], t["kv_a_norm"], t["kv_b"][1] if dense_kv_b else w["kv_b"], w["o"])
    return om.MlaOracle(c, t), dev


def cfg(**over):
    c = dict(n_embd=256, n_head=4, q_lora_rank=0, kv_lora_rank=64, qk_nope=32, qk_rope=16, v_head_dim=32,
             rms_eps=1e-6, rope_theta=10000.0, context_length=128, yarn=None)
    c.update(over)
    return c


CASES = {
    "plain_q": cfg(),
    "lora_q": cfg(q_lora_rank=96),
    "yarn": cfg(q_lora_rank=64, yarn=dict(factor=40.0, orig_context_length=64, mscale_all_dim=1.0)),
    "odd_dims": cfg(n_head=3, kv_lora_rank=96, qk_nope=24, qk_rope=6, v_head_dim=32),   # ragged latent, one head a workgroup
    "two_heads": cfg(n_head=6, kv_lora_rank=160, qk_nope=64, qk_rope=32, v_head_dim=48),
    "v3_heads": cfg(n_embd=512, n_head=16, q_lora_rank=128, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=128,
                    context_length=160),
}


@pytest.mark.parametrize("name", sorted(CASES))
def test_prefill_then_decode_matches_the_reference_graph(name):
    c = CASES[name]
    ref, dev = build(c)
    x = normal(7, (21, c["n_embd"]))
    assert close(dev.forward(x[:17], 0), ref.forward(x[:17], 0))   # prefill (causal mask)
    assert dev.cached_tokens == 17
    for p in range(17, 21):                                         # token by token
        assert close(dev.forward(x[p:p + 1], p), ref.forward(x[p:p + 1], p))
    assert dev.cached_tokens == 21


def test_prefill_equals_incremental():
    """src/quantized_deepseek2.rs:1213-1256 on the device, with its bound on the outputs."""
    c = CASES["lora_q"]
    _, a = build(c)
    _, b = build(c)
    x = normal(8, (9, c["n_embd"]))
    whole = a.forward(x, 0)
    steps = np.concatenate([b.forward(x[i:i + 1], i) for i in range(9)])
    assert np.abs(whole - steps).max() < 1e-5 * max(1.0, np.abs(whole).max())


def test_long_context_is_split_over_workgroups():
    """Enough cached tokens that a decode step splits its context (32 tokens a split or more) and the
    partial softmax results merge; scores spread over a wide range."""
    c = cfg(n_head=8, kv_lora_rank=128, qk_nope=32, qk_rope=32, v_head_dim=64, context_length=700)
    ref, dev = build(c, seed=300)
    x = normal(9, (650, c["n_embd"])) * np.float32(3.0)
    assert close(dev.forward(x[:600], 0), ref.forward(x[:600], 0))
    for p in (600, 601):
        assert close(dev.forward(x[p:p + 1], p), ref.forward(x[p:p + 1], p))
    assert close(dev.forward(x[602:650], 602), ref.forward(x[602:650], 602))  # a second prefill chunk at an offset


def test_matrix_core_attention_for_the_deepseek_geometry():
    """512 latent + 64 rope elements and heads in groups of 32 run on the f32 matrix cores: tiles of 32
    tokens, several tiles a workgroup in the prefill, several context splits in the decode steps, a
    ragged last tile."""
    c = cfg(n_embd=256, n_head=64, kv_lora_rank=512, qk_nope=32, qk_rope=64, v_head_dim=32, context_length=260)
    ref, dev = build(c, seed=700)
    x = normal(14, (250, c["n_embd"])) * np.float32(2.0)
    assert close(dev.forward(x[:150], 0), ref.forward(x[:150], 0))
    for p in (150, 151, 152):
        assert close(dev.forward(x[p:p + 1], p), ref.forward(x[p:p + 1], p))
    assert close(dev.forward(x[153:250], 153), ref.forward(x[153:250], 153))


@pytest.mark.parametrize("n_head,prompt", [(8, 1), (8, 14), (24, 159), (32, 317)])
def test_one_token_over_a_short_context(n_head, prompt):
    """Steps in which a wave takes two heads and 16 cached tokens: contexts of one token, around whole runs of 16, and over the
    line to the matrix-core kernel."""
    c = cfg(n_embd=256, n_head=n_head, kv_lora_rank=512, qk_nope=64, qk_rope=64, v_head_dim=32, context_length=prompt + 8)
    ref, dev = build(c, seed=750 + n_head)
    x = normal(18, (prompt + 5, c["n_embd"])) * np.float32(2.0)
    assert close(dev.forward(x[:prompt], 0), ref.forward(x[:prompt], 0))
    for p in range(prompt, prompt + 5):
        assert close(dev.forward(x[p:p + 1], p), ref.forward(x[p:p + 1], p), 1e-4), p


@pytest.mark.parametrize("n_head,steps", [(3, (47, 48, 129, 1)), (8, (160, 95, 48)), (16, (33, 127, 2))])
def test_many_tokens_over_keys_and_values_per_head(n_head, steps):
    """DeepSeek's head sizes from 48 tokens a call on: the cached latents expanded to keys and values, attention on split
    f16 operands; calls below and above the line in turn, head counts that are no multiple of 8, part tiles of keys and
    tokens, and inputs whose size (and with it the unnormed rope keys') differs a thousandfold between tokens."""
    c = cfg(n_embd=256, n_head=n_head, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=128, context_length=320)
    ref, dev = build(c, seed=800 + n_head)
    total = sum(steps)
    x = normal(15, (total, c["n_embd"])) * np.exp(np.linspace(-5.0, 2.0, total)[np.random.default_rng(3).permutation(total)])[:, None]
    x, pos = x.astype(np.float32), 0
    for n in steps:
        assert close(dev.forward(x[pos:pos + n], pos), ref.forward(x[pos:pos + n], pos)), (pos, n)
        pos += n


@pytest.mark.parametrize("zero", ["queries and up-projection", "queries", "keys of the up-projection", "rope keys and queries"])
def test_heads_whose_queries_or_keys_are_zero(zero):
    """48 tokens a call and more, where a score is the sum of two products that each have scales of their own: heads of zeros
    (pruned or padded ones) in every place, beside heads with values.  Head 1 has the zeros, head 2 keeps all."""
    c = cfg(n_embd=256, n_head=3, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=128, context_length=160)
    ref, _ = build(c, seed=860)
    rows = {n: (256 if n != "kv_b" else 512, np.asarray(ref.t[n][1]).view(np.uint8)) for n in ("q", "kv_a_mqa", "kv_b", "o")}
    shape = {"q": (576, 256), "kv_a_mqa": (576, 256), "kv_b": (768, 512), "o": (256, 384)}
    raw = {n: rows[n][1].reshape(shape[n][0], -1).copy() for n in rows}
    if "queries" in zero:
        raw["q"][192 + (128 if "rope" in zero else 0):192 + (192 if "rope" in zero or "up" in zero else 128)] = 0
    if "up-projection" in zero:
        raw["kv_b"][256:256 + (256 if "queries" in zero else 128)] = 0
    if "rope keys" in zero:
        raw["kv_a_mqa"][512:] = 0
    t = dict(ref.t, **{n: (capi.Q8_0, b.reshape(-1)) for n, b in raw.items()})
    w = {n: capi.Weight.upload(capi.Q8_0, raw[n].reshape(-1), *shape[n]) for n in raw}
    mc = capi.MlaConfig(n_embd=256, n_head=3, q_lora_rank=0, kv_lora_rank=512, qk_nope_head_dim=128, qk_rope_head_dim=64,
                        v_head_dim=128, n_ctx=160, rms_eps=1e-6, rope_theta=1e4)
    dev, want = capi.Mla(mc, w["q"], w["kv_a_mqa"], t["kv_a_norm"], w["kv_b"], w["o"]), om.MlaOracle(c, t)
    x = normal(19, (130, 256))
    assert close(dev.forward(x[:64], 0), want.forward(x[:64], 0))
    assert close(dev.forward(x[64:], 64), want.forward(x[64:], 64))


def f16(x):
    return x.astype(np.float16).astype(np.float64)


def test_many_tokens_hold_every_operand_to_more_than_f16():
    """Latent attention of 200 tokens against 64 bits.  The inputs are unit vectors, so that the products in front of the attention
    are columns of their weights, and the error is the attention's and that of the 16-bit activations of the product behind it:
    half a step of 2^-15 of the largest of 256, 0.9e-5 of the norm for values of which that is 3 times the rest.  An operand
    that was held to f16 alone would show: each is rounded in turn here, on the CPU, and is twice over the bound or more."""
    nh, S, rng = 2, 200, np.random.default_rng(6)
    shape = {"q": (nh * 192, 256), "kv_a": (576, 256), "kv_b": (nh * 256, 512), "o": (256, nh * 128)}
    sigma = {"q": 2.0, "kv_a": 1.0, "kv_b": 0.05, "o": 0.1}
    blocks = {n: quantized(capi.Q8_0, 880 + i, *shape[n], sigma[n]) for i, n in enumerate(sorted(shape))}
    W = {n: oracle.dequantize(capi.Q8_0, b).reshape(shape[n]).astype(np.float64) for n, b in blocks.items()}
    w = {n: capi.Weight.upload(capi.Q8_0, b, *shape[n]) for n, b in blocks.items()}
    norm = (1.0 + 0.1 * normal(890, (512,))).astype(np.float32)
    mc = capi.MlaConfig(n_embd=256, n_head=nh, q_lora_rank=0, kv_lora_rank=512, qk_nope_head_dim=128, qk_rope_head_dim=64,
                        v_head_dim=128, n_ctx=256, rms_eps=1e-6, rope_theta=1e4)
    idx = rng.permutation(256)[:S]
    got = capi.Mla(mc, w["q"], w["kv_a"], norm, w["kv_b"], w["o"]).forward(np.eye(256, dtype=np.float32)[idx], 0)

    angle = np.arange(S)[:, None] * 1e4 ** (-np.arange(0, 64, 2) / 64.0)
    turn = lambda v: np.stack([v[..., 0::2] * np.cos(angle) - v[..., 1::2] * np.sin(angle),
                               v[..., 1::2] * np.cos(angle) + v[..., 0::2] * np.sin(angle)], -1).reshape(v.shape)
    q, comp = W["q"][:, idx].T.reshape(S, nh, 192), W["kv_a"][:, idx].T
    lat = comp[:, :512] / np.sqrt((comp[:, :512] ** 2).mean(1, keepdims=True) + 1e-6) * norm
    kpe, up = turn(comp[:, 512:]), W["kv_b"].reshape(nh, 2, 128, 512)

    def block(**rounded):
        as_is = lambda v: v
        r = {n: rounded.get(n, as_is) for n in ("latents", "up", "queries", "rope", "keys", "values", "weights")}
        ctx = []
        for h in range(nh):
            k, v = (r["latents"](lat) @ r["up"](u).T for u in up[h])
            s = r["queries"](q[:, h, :128]) @ r["keys"](k).T + r["queries"](turn(q[:, h, 128:])) @ r["rope"](kpe).T
            s = np.where(np.tri(S, dtype=bool), s / np.sqrt(192.0), -np.inf)
            e = np.exp(s - s.max(1, keepdims=True))
            ctx.append(r["weights"](e) @ r["values"](v) / e.sum(1, keepdims=True))
        return np.concatenate(ctx, 1) @ W["o"].T

    want = block()
    err = lambda y: np.linalg.norm(y - want) / np.linalg.norm(want)
    assert err(got) < 3e-5, err(got)
    for n in ("latents", "up", "queries", "rope", "keys", "values", "weights"):
        assert err(block(**{n: f16})) > 8e-5, (n, err(block(**{n: f16})))


@pytest.mark.parametrize("value", [np.nan, np.inf])
@pytest.mark.parametrize("at", [0, 40, 63])
def test_a_token_that_is_not_finite_stays_out_of_those_in_front(at, value):
    """64 tokens a call, whose tiles of 32 keys hold tokens of which some queries see only a part: a token of NaNs is in the
    results of those behind it, in this call and the next, and in none in front."""
    c = cfg(n_embd=256, n_head=3, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=128, context_length=160)
    ref, dev = build(c, seed=870)
    x = normal(20, (128, 256))
    want = ref.forward(x[:64], 0)
    x[at, 7] = value
    got = dev.forward(x[:64], 0)
    assert close(got[:at], want[:at])
    assert not np.isfinite(got[at:]).any(axis=1).any()
    assert not np.isfinite(dev.forward(x[64:], 64)).any()


def test_heads_in_groups_where_their_keys_and_values_exceed_the_buffer():
    """256 heads of 4200 tokens are expanded in three groups (512 MiB of keys and values each at most).  The 256 are 32
    copies of 8 and so are the output projection's columns: the sum is 32 times what the 8 alone give, up to the order of
    the additions."""
    c8 = cfg(n_embd=256, n_head=8, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=128, context_length=4224)
    t8, few = build(c8, seed=900)
    t8 = t8.t
    raw = lambda name, rows: np.asarray(t8[name][1]).view(np.uint8).reshape(rows, -1)
    q = np.tile(raw("q", 8 * 192), (32, 1))
    kv_b = np.tile(raw("kv_b", 8 * 256), (32, 1))
    o = np.tile(raw("o", 256), (1, 32))
    w = {n: capi.Weight.upload(capi.Q8_0, np.ascontiguousarray(b), r, k)
         for n, b, r, k in (("q", q, 256 * 192, 256), ("kv_a", raw("kv_a_mqa", 576), 576, 256), ("kv_b", kv_b, 65536, 512), ("o", o, 256, 32768))}
    mc = capi.MlaConfig(n_embd=256, n_head=256, q_lora_rank=0, kv_lora_rank=512, qk_nope_head_dim=128, qk_rope_head_dim=64,
                        v_head_dim=128, n_ctx=4224, rms_eps=1e-6, rope_theta=1e4)
    many = capi.Mla(mc, w["q"], w["kv_a"], t8["kv_a_norm"], w["kv_b"], w["o"])
    x = normal(16, (4200, 256))
    a, b = few.forward(x, 0), many.forward(x, 0) / 32
    assert np.abs(a - b).max() < 3e-4 * max(1.0, np.abs(a).max())


def test_many_tokens_where_expanding_stops_paying():
    """64 tokens of 128 heads behind 10000 others are absorbed again (keys and values of two groups of heads would be expanded,
    each walked by half as many workgroups as there are compute units), and 64 behind 600 are not.  Columns of 32 copies of 4
    heads, as above: against an object of those 4, which expands in both places."""
    c4 = cfg(n_embd=256, n_head=4, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=128, context_length=10112)
    t4, few = build(c4, seed=920)
    raw = lambda name, rows: np.asarray(t4.t[name][1]).view(np.uint8).reshape(rows, -1)
    w = {n: capi.Weight.upload(capi.Q8_0, np.ascontiguousarray(b), r, k)
         for n, b, r, k in (("q", np.tile(raw("q", 768), (32, 1)), 128 * 192, 256), ("kv_a", raw("kv_a_mqa", 576), 576, 256),
                            ("kv_b", np.tile(raw("kv_b", 1024), (32, 1)), 32768, 512), ("o", np.tile(raw("o", 256), (1, 32)), 256, 16384))}
    mc = capi.MlaConfig(n_embd=256, n_head=128, q_lora_rank=0, kv_lora_rank=512, qk_nope_head_dim=128, qk_rope_head_dim=64,
                        v_head_dim=128, n_ctx=10112, rms_eps=1e-6, rope_theta=1e4)
    many = capi.Mla(mc, w["q"], w["kv_a"], t4.t["kv_a_norm"], w["kv_b"], w["o"])
    x, pos = normal(22, (10112, 256)), 0
    for n in (600, 64, 9384, 64):
        a, b = few.forward(x[pos:pos + n], pos), many.forward(x[pos:pos + n], pos) / 32
        assert np.abs(a - b).max() < 3e-4 * max(1.0, np.abs(a).max()), pos
        pos += n


def test_a_capture_of_the_first_call_that_would_expand():
    """64 tokens of 128 heads behind 10000 others are absorbed, so an object that has seen only such calls and shorter ones holds no
    buffer for expanded keys and values, and none can be had while a graph is captured: 64 tokens at the front are then absorbed
    too.  The graph replays to what an object of 4 of the heads gives (columns of 32 copies, as above), with eager work between."""
    import torch
    c4 = cfg(n_embd=256, n_head=4, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=128, context_length=10112)
    t4, few = build(c4, seed=930)
    raw = lambda name, rows: np.asarray(t4.t[name][1]).view(np.uint8).reshape(rows, -1)
    w = {n: capi.Weight.upload(capi.Q8_0, np.ascontiguousarray(b), r, k)
         for n, b, r, k in (("q", np.tile(raw("q", 768), (32, 1)), 128 * 192, 256), ("kv_a", raw("kv_a_mqa", 576), 576, 256),
                            ("kv_b", np.tile(raw("kv_b", 1024), (32, 1)), 32768, 512), ("o", np.tile(raw("o", 256), (1, 32)), 256, 16384))}
    mc = capi.MlaConfig(n_embd=256, n_head=128, q_lora_rank=0, kv_lora_rank=512, qk_nope_head_dim=128, qk_rope_head_dim=64,
                        v_head_dim=128, n_ctx=10112, rms_eps=1e-6, rope_theta=1e4)
    many = capi.Mla(mc, w["q"], w["kv_a"], t4.t["kv_a_norm"], w["kv_b"], w["o"])
    x = torch.from_numpy(normal(23, (64, 256))).cuda()
    y = torch.zeros(64, 256, device="cuda")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()
    with torch.cuda.stream(stream):
        for n in [40] * 250 + [64]:
            many.forward_dev(n, many.cached_tokens, x.data_ptr(), y.data_ptr(), stream.cuda_stream)
        stream.synchronize()
        many.reset()
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            many.forward_dev(64, 0, x.data_ptr(), y.data_ptr(), torch.cuda.current_stream().cuda_stream)
        want = few.forward(x.cpu().numpy(), 0)
        for rep in range(3):
            y.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            got = y.cpu().numpy() / 32
            assert np.abs(got - want).max() < 3e-4 * max(1.0, np.abs(want).max()), rep
    del graph
    torch.cuda.synchronize()
    capi.stream_release(stream.cuda_stream)


def test_memory_of_an_object_over_a_long_context():
    """Keys and values of 128 heads over 16384 positions would be 2 GiB, and 512 MiB are taken; beside them 130 MB of the
    up-projection as f32 and as operands, 75 of the cache and its copy as operands, and 60 of scratch."""
    import torch
    w = {n: capi.Weight.upload(capi.Q8_0, quantized(capi.Q8_0, 910 + i, r, k), r, k)
         for i, (n, r, k) in enumerate((("q", 128 * 192, 256), ("kv_a", 576, 256), ("kv_b", 32768, 512), ("o", 256, 16384)))}
    mc = capi.MlaConfig(n_embd=256, n_head=128, q_lora_rank=0, kv_lora_rank=512, qk_nope_head_dim=128, qk_rope_head_dim=64,
                        v_head_dim=128, n_ctx=16384, rms_eps=1e-6, rope_theta=1e4)
    before = torch.cuda.mem_get_info()[0]
    dev = capi.Mla(mc, w["q"], w["kv_a"], np.ones(512, np.float32), w["kv_b"], w["o"])
    dev.forward(normal(21, (64, 256)), 0)
    assert before - torch.cuda.mem_get_info()[0] < 900 << 20


@pytest.mark.parametrize("n_head,vh,prompt", [(4, 64, 1), (4, 128, 300), (32, 128, 40), (32, 64, 700)])
def test_one_token_over_q4k_blocks_of_the_up_projection(n_head, vh, prompt):
    """Single-token steps that read kv_b as Q4_K blocks (512 latents, 128 unrotated elements a head), against the same layer
    over its f32 values: short contexts, which take one launch between the query and the output projection, value rows of one and two
    workgroups a head.  The same weights up to the order of f32 sums of 128 and 512 terms and of their offsets: 1e-5 of the largest."""
    c = cfg(n_embd=256, n_head=n_head, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=vh, context_length=prompt + 8)
    ref, dev = build(c, qtype=capi.Q4_K, seed=450 + n_head)
    raw = {n: (r, k) for n, r, k in (("q", n_head * 192, 256), ("kv_a_mqa", 576, 256), ("o", 256, n_head * vh))}
    w = {n: capi.Weight.upload(capi.Q4_K, ref.t[n][1], r, k) for n, (r, k) in raw.items()}
    mc = capi.MlaConfig(n_embd=256, n_head=n_head, q_lora_rank=0, kv_lora_rank=512, qk_nope_head_dim=128, qk_rope_head_dim=64,
                        v_head_dim=vh, n_ctx=prompt + 8, rms_eps=1e-6, rope_theta=1e4)
    values = oracle.dequantize(capi.Q4_K, ref.t["kv_b"][1]).reshape(n_head * (128 + vh), 512).astype(np.float32)
    dense = capi.Mla(mc, w["q"], w["kv_a_mqa"], ref.t["kv_a_norm"], values, w["o"])
    x = normal(17, (prompt + 3, 256)) * np.float32(2.0)
    dev.forward(x[:prompt], 0), dense.forward(x[:prompt], 0)
    for p in range(prompt, prompt + 3):
        a, b = dev.forward(x[p:p + 1], p), dense.forward(x[p:p + 1], p)
        assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max(), p


@pytest.mark.parametrize("n_head,vh,prompt", [(4, 128, 894), (32, 64, 894), (32, 128, 1500), (128, 128, 893), (264, 64, 5), (136, 128, 318), (160, 128, 318)])
def test_steps_in_three_launches_over_q4k_blocks(n_head, vh, prompt):
    """As above, absorption, attention and merging with the value rows a launch each: from 896 cached tokens on (the first steps of some cases
    are still one launch), by either attention kernel, and with more heads times 64 value rows than compute units, where the attention of up
    to 320 tokens has a kernel of its own."""
    c = cfg(n_embd=256, n_head=n_head, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=vh, context_length=prompt + 8)
    ref, dev = build(c, qtype=capi.Q4_K, seed=460 + n_head)
    raw = {n: (r, k) for n, r, k in (("q", n_head * 192, 256), ("kv_a_mqa", 576, 256), ("o", 256, n_head * vh))}
    w = {n: capi.Weight.upload(capi.Q4_K, ref.t[n][1], r, k) for n, (r, k) in raw.items()}
    mc = capi.MlaConfig(n_embd=256, n_head=n_head, q_lora_rank=0, kv_lora_rank=512, qk_nope_head_dim=128, qk_rope_head_dim=64,
                        v_head_dim=vh, n_ctx=prompt + 8, rms_eps=1e-6, rope_theta=1e4)
    values = oracle.dequantize(capi.Q4_K, ref.t["kv_b"][1]).reshape(n_head * (128 + vh), 512).astype(np.float32)
    dense = capi.Mla(mc, w["q"], w["kv_a_mqa"], ref.t["kv_a_norm"], values, w["o"])
    x = normal(18, (prompt + 6, 256)) * np.float32(2.0)
    dev.forward(x[:prompt], 0), dense.forward(x[:prompt], 0)
    for p in range(prompt, prompt + 6):
        a, b = dev.forward(x[p:p + 1], p), dense.forward(x[p:p + 1], p)
        assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max(), p


@pytest.mark.parametrize("n_head,vh,prompt", [(4, 64, 0), (2, 128, 14), (4, 192, 126), (128, 128, 253), (4, 64, 893)])
def test_a_step_in_one_launch_over_q4k_blocks(n_head, vh, prompt):
    """Steps of one launch between the query and the output projection: an empty cache, around a wave's turn (16 tokens), a run of
    all waves' (128), two of them, and the line to the launches of long contexts (896); few heads, as many workgroups as compute units.
    The cache that the steps leave is read by a call of two tokens, which has other kernels.  1e-5 of the largest as above."""
    c = cfg(n_embd=256, n_head=n_head, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=vh, context_length=prompt + 8)
    ref, dev = build(c, qtype=capi.Q4_K, seed=470 + n_head)
    raw = {n: (r, k) for n, r, k in (("q", n_head * 192, 256), ("kv_a_mqa", 576, 256), ("o", 256, n_head * vh))}
    w = {n: capi.Weight.upload(capi.Q4_K, ref.t[n][1], r, k) for n, (r, k) in raw.items()}
    mc = capi.MlaConfig(n_embd=256, n_head=n_head, q_lora_rank=0, kv_lora_rank=512, qk_nope_head_dim=128, qk_rope_head_dim=64,
                        v_head_dim=vh, n_ctx=prompt + 8, rms_eps=1e-6, rope_theta=1e4)
    values = oracle.dequantize(capi.Q4_K, ref.t["kv_b"][1]).reshape(n_head * (128 + vh), 512).astype(np.float32)
    dense = capi.Mla(mc, w["q"], w["kv_a_mqa"], ref.t["kv_a_norm"], values, w["o"])
    x = normal(19, (prompt + 8, 256)) * np.float32(2.0)
    if prompt:
        dev.forward(x[:prompt], 0), dense.forward(x[:prompt], 0)
    for p in range(prompt, prompt + 6):
        a, b = dev.forward(x[p:p + 1], p), dense.forward(x[p:p + 1], p)
        assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max(), p
    a, b = dev.forward(x[prompt + 6:], prompt + 6), dense.forward(x[prompt + 6:], prompt + 6)
    assert np.abs(a - b).max() <= 1e-5 * np.abs(b).max()


def test_dense_kv_b_and_other_formats():
    c = cfg(kv_lora_rank=256, n_embd=256, v_head_dim=64)
    for qtype in (capi.Q4_K, capi.Q6_K):
        ref, dev = build(c, qtype=qtype, seed=400 + qtype)
        x = normal(10, (5, c["n_embd"]))
        assert close(dev.forward(x, 0), ref.forward(x, 0))
    ref, dev = build(cfg(), dense_kv_b=True, seed=500)
    x = normal(11, (6, 256))
    assert close(dev.forward(x, 0), ref.forward(x, 0))
    # the latent width of the reference's own tiny attention (src/quantized_deepseek2.rs:1102-1125)
    c = cfg(n_embd=32, n_head=2, kv_lora_rank=6, qk_nope=4, qk_rope=4, v_head_dim=16)
    ref, dev = build(c, dense_kv_b=True, seed=600)
    x = normal(12, (4, 32))
    assert close(dev.forward(x[:3], 0), ref.forward(x[:3], 0))
    assert close(dev.forward(x[3:], 3), ref.forward(x[3:], 3))


def test_reset_and_position_checks():
    c = CASES["plain_q"]
    ref, dev = build(c)
    x = normal(12, (4, c["n_embd"]))
    first = dev.forward(x, 0)
    with pytest.raises(capi.JoshuaHipError, match="tokens are cached"):
        dev.forward(x[:1], 0)
    dev.reset()
    assert dev.cached_tokens == 0
    assert np.array_equal(dev.forward(x, 0), first)
    with pytest.raises(capi.JoshuaHipError, match="exceed the context"):
        dev.forward(normal(13, (c["context_length"], c["n_embd"])), 4)


def test_create_rejects_wrong_shapes():
    c = CASES["plain_q"]
    blocks = quantized(capi.Q8_0, 1, 64, 256)
    w = capi.Weight.upload(capi.Q8_0, blocks, 64, 256)
    mc = capi.MlaConfig(n_embd=256, n_head=4, q_lora_rank=0, kv_lora_rank=64, qk_nope_head_dim=32, qk_rope_head_dim=16,
                        v_head_dim=32, n_ctx=16, rms_eps=1e-6, rope_theta=1e4)
    with pytest.raises(capi.JoshuaHipError, match="attn_q is"):
        capi.Mla(mc, w, w, np.ones(64, np.float32), w, w)


@pytest.mark.parametrize("n_head", [3, 32])
def test_calls_add_to_the_keys_and_values_of_earlier_ones(n_head):
    """Calls of many tokens expand those since the last such call only, short ones in between (absorbed) and part-filled tiles of
    32 tokens among them; after a reset other tokens take all places."""
    c = cfg(n_embd=256, n_head=n_head, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=128, context_length=640)
    ref, dev = build(c, seed=940)
    for seed, steps in ((24, (50, 1, 1, 64, 100, 3, 49, 200)), (25, (48, 47, 96, 160)), (26, (40, 33, 130))):
        x, pos = normal(seed, (sum(steps), 256)), 0
        for n in steps:
            assert close(dev.forward(x[pos:pos + n], pos), ref.forward(x[pos:pos + n], pos)), (steps, pos)
            pos += n
        dev.reset()
        ref, _ = build(c, seed=940)


def test_a_captured_call_behind_tokens_that_were_not_expanded():
    """64 tokens behind 100 that the call before expanded are captured; the graph is replayed behind 100 others that short, absorbed
    calls wrote, and so were never expanded."""
    import torch
    c = cfg(n_embd=256, n_head=4, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=128, context_length=192)
    _, dev = build(c, seed=950)
    _, fresh = build(c, seed=950)
    a, b = (torch.from_numpy(normal(seed, (100, 256))).cuda() for seed in (27, 28))
    x = torch.from_numpy(normal(29, (64, 256))).cuda()
    y, rest = torch.zeros(64, 256, device="cuda"), torch.zeros(100, 256, device="cuda")
    stream = torch.cuda.Stream()
    torch.cuda.synchronize()

    def run(m, t, steps):
        m.reset()
        for n in steps:
            p = m.cached_tokens
            m.forward_dev(n, p, t.data_ptr() + 1024 * p, rest.data_ptr(), stream.cuda_stream)

    with torch.cuda.stream(stream):
        run(dev, a, (100,))
        dev.forward_dev(64, 100, x.data_ptr(), y.data_ptr(), stream.cuda_stream)
        stream.synchronize()
        run(dev, a, (100,))
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph, stream=stream):
            dev.forward_dev(64, 100, x.data_ptr(), y.data_ptr(), torch.cuda.current_stream().cuda_stream)
        for t, steps in ((a, (100,)), (b, (40, 40, 20)), (b, (100,)), (a, (30, 30, 40))):
            run(fresh, t, steps)
            want = fresh.forward(x.cpu().numpy(), 100)
            run(dev, t, steps)
            y.fill_(float("nan"))
            graph.replay()
            torch.cuda.synchronize()
            assert np.abs(y.cpu().numpy() - want).max() < 3e-4 * max(1.0, np.abs(want).max()), steps
    del graph
    torch.cuda.synchronize()
    capi.stream_release(stream.cuda_stream)


def test_one_token_whose_query_norm_rides_in_the_product():
    """A Q4_K query up-projection of 1536 columns: RMSNorm and product of a single token are one launch; several tokens, and other
    formats, take two."""
    c = cfg(n_embd=256, n_head=4, q_lora_rank=1536, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=128)
    for qtype in (capi.Q4_K, capi.Q8_0):
        ref, dev = build(c, qtype=qtype, seed=960)
        x, pos = normal(30, (12, 256)), 0
        for n in (3, 1, 1, 6, 1):
            assert close(dev.forward(x[pos:pos + n], pos), ref.forward(x[pos:pos + n], pos)), (qtype, pos)
            pos += n


@pytest.mark.parametrize("n_head", [96, 100])
def test_a_query_norm_in_front_of_one_and_two_tiles_a_workgroup(n_head):
    """1152 and 1200 tiles of 16 rows of 1536 columns."""
    c = cfg(n_embd=256, n_head=n_head, q_lora_rank=1536, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=64)
    ref, dev = build(c, qtype=capi.Q4_K, seed=970)
    x, pos = normal(31, (5, 256)), 0
    for n in (3, 1, 1):
        assert close(dev.forward(x[pos:pos + n], pos), ref.forward(x[pos:pos + n], pos)), pos
        pos += n


def test_query_and_latent_down_projections_as_one_product():
    """256 tokens over 4096 columns take q_a and kv_a as one product, 96 take two: both between single tokens, which take one."""
    c = cfg(n_embd=4096, n_head=2, q_lora_rank=256, kv_lora_rank=512, qk_nope=128, qk_rope=64, v_head_dim=128, context_length=640)
    ref, dev = build(c, seed=970)
    x, pos = normal(31, (620, 4096)), 0
    for n in (256, 1, 96, 1, 257, 9):
        assert close(dev.forward(x[pos:pos + n], pos), ref.forward(x[pos:pos + n], pos)), pos
        pos += n
