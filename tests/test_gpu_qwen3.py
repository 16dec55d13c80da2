"""End-to-end dense Qwen3 decode on the device against the numpy graph over the
oracle matmul: teacher-forced logits after a prefill and on every decode step,
the KV-cache position contract, and the greedy pick's tie order."""
import numpy as np
import pytest

import oracle
from oracle import qwen3 as oq
from joshua_amd import capi, synth
from joshua_amd.synth.model import qwen3_tensor_plan, qwen3_tensors
from tests.h6_swiglu import swiglu_product

pytestmark = pytest.mark.gpu

CFG = dict(n_layer=3, hidden=512, n_head=4, n_kv_head=2, head_dim=64, ffn=1024, vocab=768, n_ctx=48,
           rms_eps=1e-6, rope_theta=1e6)


def make(cfg, seed, mix="q4_k_m", override=None):
    tensors = {n: (qt, d) for n, qt, d in qwen3_tensors(cfg, seed, mix)}
    if override:
        tensors.update(override)
    c = capi.Qwen3Config(cfg["n_layer"], cfg["hidden"], cfg["n_head"], cfg["n_kv_head"], cfg["head_dim"], cfg["ffn"],
                         cfg["vocab"], cfg["n_ctx"], cfg["rms_eps"], cfg["rope_theta"])
    m = capi.Qwen3(c)
    for n, (qt, d) in tensors.items():
        m.set_tensor(n, qt, d)
    return m, oq.Qwen3Oracle(cfg, tensors, avx2=oracle.have_avx2())


def close(got, ref, tol=1e-3):
    # the bound the reference's acceptance uses for f32 results: |gpu - ref| <= tol * max(|ref|, 1)
    err = np.abs(got - ref) / np.maximum(np.abs(ref), 1.0)
    return float(err.max()) <= tol, float(err.max())


@pytest.mark.parametrize("mix", ["q4_k_m", "8"])
def test_teacher_forced_logits(mix):
    m, o = make(CFG, 21, mix)
    prompt = [3, 700, 41, 41, 256, 9, 88, 511, 2, 640, 77]
    got, ref = m.forward(prompt, 0), o.forward(prompt, 0)
    ok, e = close(got, ref)
    assert ok, f"prefill: {e}"
    pos = len(prompt)
    for t in [5, 123, 767, 0, 350, 12]:
        got, ref = m.forward([t], pos), o.forward([t], pos)
        ok, e = close(got, ref)
        assert ok, f"pos {pos}: {e}"
        g = m.greedy()
        top2 = np.sort(ref)[-2:]
        if top2[1] - top2[0] > 2e-3 * max(abs(top2[1]), 1.0):
            assert g == oq.greedy(ref)
        assert got[g] == got.max()
        pos += 1


@pytest.mark.parametrize("mix", ["q4_k_m", "q4_k"])
def test_single_token_steps_with_4096_wide_rows(mix):
    """hidden = 4096: a single-token step runs residual add + RMSNorm + q|k(|v) and + gate|up as
    one launch each ("q4_k": every matrix Q4_K, v inside the fused launch; "q4_k_m": some layers keep
    attn_v as Q6_K, a launch of its own over the normalised row the fused kernel leaves behind)."""
    cfg = dict(CFG, n_layer=4, hidden=4096, n_head=4, n_kv_head=2, head_dim=128, ffn=1024, vocab=512, n_ctx=32)
    m, o = make(cfg, 29, mix)
    prompt = [3, 500, 41, 41, 256, 9]
    ok, e = close(m.forward(prompt, 0), o.forward(prompt, 0))
    assert ok, f"prefill: {e}"
    pos = len(prompt)
    for t in [5, 123, 511, 0, 350]:
        ok, e = close(m.forward([t], pos), o.forward([t], pos))
        assert ok, f"pos {pos}: {e}"
        pos += 1


@pytest.mark.parametrize("mix", ["q4_k_m", "q4_k"])
def test_single_token_steps_with_2048_wide_rows(mix):
    """hidden = 2048: residual add + RMSNorm + q|k(|v) of a single-token step are one launch of the kernel
    that takes a tile of 16 rows a workgroup; gate, up and the rest run as launches of their own."""
    cfg = dict(CFG, n_layer=4, hidden=2048, n_head=4, n_kv_head=2, head_dim=128, ffn=768, vocab=512, n_ctx=32)
    m, o = make(cfg, 37, mix)
    prompt = [3, 500, 41, 41, 256, 9]
    ok, e = close(m.forward(prompt, 0), o.forward(prompt, 0))
    assert ok, f"prefill: {e}"
    pos = len(prompt)
    for t in [5, 123, 511, 0, 350]:
        ok, e = close(m.forward([t], pos), o.forward([t], pos))
        assert ok, f"pos {pos}: {e}"
        pos += 1


def test_single_token_steps_with_attn_v_of_another_format_in_the_qk_launch():
    """hidden = 4096 and 2560 rows of q|k: on the layers that keep attn_v as Q6_K or Q8_0 (four of these eight, two of
    each) its tiles run in the launch of residual add + RMSNorm + q|k, behind the workgroups of the Q4_K product."""
    cfg = dict(CFG, n_layer=8, hidden=4096, n_head=16, n_kv_head=4, head_dim=128, ffn=512, vocab=512, n_ctx=32)
    m, o = make(cfg, 39, "q4_k_m")
    kinds = {o.t[f"blk.{l}.attn_v.weight"][0] for l in range(8)}
    assert {capi.Q6_K, capi.Q8_0} <= kinds
    prompt = [3, 500, 41, 41, 256, 9]
    ok, e = close(m.forward(prompt, 0), o.forward(prompt, 0))
    assert ok, f"prefill: {e}"
    pos = len(prompt)
    for t in [5, 123, 511, 0]:
        ok, e = close(m.forward([t], pos), o.forward([t], pos))
        assert ok, f"pos {pos}: {e}"
        pos += 1


def test_single_token_steps_over_one_to_eighteen_key_chunks():
    """32 heads of 128, four KV heads: single-token steps whose split attention covers one, two, three, five and
    eighteen chunks of 64 keys, between prefill chunks of 61 to 830 tokens."""
    cfg = dict(CFG, n_layer=2, hidden=512, n_head=32, n_kv_head=4, head_dim=128, ffn=512, vocab=512, n_ctx=1120)
    m, o = make(cfg, 41, "q4_k")
    rng = np.random.default_rng(17)
    toks = [int(t) for t in rng.integers(0, cfg["vocab"], size=1110)]
    pos = 0
    for step in (1, 1, 61, 1, 1, 1, 64, 1, 130, 1, 1, 830, 1, 1):   # single-token steps at 1, 2, 64..66, 131, 262, 1093.. cached tokens
        chunk = toks[pos:pos + step]
        ok, e = close(m.forward(chunk, pos), o.forward(chunk, pos))
        assert ok, f"pos {pos} +{step}: {e}"
        pos += step


def test_paired_gate_up_rows_serve_prefill_and_replacement():
    """With 4096-wide Q4_K rows the gate and up matrices are stored with alternating rows (the
    single-token launch applies SwiGLU itself); multi-token steps read them as strided views, and a
    replaced part sends the layer back to separate launches."""
    cfg = dict(CFG, n_layer=2, hidden=4096, n_head=4, n_kv_head=2, head_dim=128, ffn=512, vocab=512, n_ctx=40)
    m, o = make(cfg, 31, "q4_k")
    toks = [7, 400, 41, 300, 256, 9, 12, 13, 14, 15, 16, 17, 18, 19, 20, 21, 22, 23, 24, 25]
    ok, e = close(m.forward(toks[:1], 0), o.forward(toks[:1], 0))      # fuses on the first single-token step
    assert ok, e
    ok, e = close(m.forward(toks[1:4], 1), o.forward(toks[1:4], 1))    # 3 rows: views under the few-row kernel
    assert ok, e
    ok, e = close(m.forward(toks[4:], 4), o.forward(toks[4:], 4))      # 16 rows
    assert ok, e
    m.reset(), o.reset()
    ok, e = close(m.forward(toks + toks, 0), o.forward(toks + toks, 0))  # 40 rows: views under the GEMM
    assert ok, e
    name = "blk.1.ffn_up.weight"
    tensors = {n: (qt, d) for n, qt, d in qwen3_tensors(cfg, 31, "q4_k")}
    tensors[name] = {n: (qt, d) for n, qt, d in qwen3_tensors(cfg, 99, "q4_k")}[name]
    m.set_tensor(name, *tensors[name])
    o2 = oq.Qwen3Oracle(cfg, tensors, avx2=oracle.have_avx2())
    m.reset()
    ok, e = close(m.forward([5], 0), o2.forward([5], 0))
    assert ok, e
    ok, e = close(m.forward([6], 1), o2.forward([6], 1))
    assert ok, e


@pytest.mark.parametrize("qtype", [capi.Q8_0, capi.Q6_K, capi.Q4_1, capi.MXFP4])
def test_short_steps_over_embeddings_of_any_format(qtype):
    """Steps of up to eight tokens gather their rows in the launch that makes the angles, nine in launches of their own; first and last
    rows of the table, a token twice."""
    count = CFG["vocab"] * CFG["hidden"]
    blocks = synth.random_blocks(qtype, 61, count) if qtype in capi.GENERIC_TYPES else synth.normal_quantized(qtype, 61, count, 1.0)
    m, o = make(CFG, 62, override={"token_embd.weight": (qtype, blocks)})
    pos = 0
    for tokens in ([0], [767, 5], [3, 3, 700, 41, 256, 9, 88], [767, 0, 41, 41, 256, 9, 88, 511], [2, 640, 77, 5, 9, 1, 766, 4, 4], [123]):
        ok, e = close(m.forward(tokens, pos), o.forward(tokens, pos))
        assert ok, f"{len(tokens)} tokens at {pos}: {e}"
        pos += len(tokens)


def test_prefill_in_two_chunks_matches_one():
    m, o = make(CFG, 22)
    toks = list(range(10, 30))
    ref = o.forward(toks, 0)
    m.forward(toks[:13], 0)
    got = m.forward(toks[13:], 13)
    ok, e = close(got, ref)
    assert ok, e


@pytest.mark.parametrize("n_head,n_kv", [(4, 1), (4, 2), (2, 2)])
def test_prefill_in_chunks_with_head_size_128(n_head, n_kv):
    """Chunks of more than 8 tokens at a position past 0: the tiled attention with keys already in the
    cache, token counts that leave the last tile part empty, and a chunk that starts inside a key tile."""
    cfg = dict(CFG, n_ctx=96, n_layer=2, head_dim=128, n_head=n_head, n_kv_head=n_kv)
    m, o = make(cfg, 27)
    rng = np.random.default_rng(4)
    toks = [int(t) for t in rng.integers(0, cfg["vocab"], size=90)]
    pos = 0
    for step in (21, 16, 37, 9):
        chunk = toks[pos:pos + step]
        ok, e = close(m.forward(chunk, pos), o.forward(chunk, pos))
        assert ok, f"pos {pos} +{step}: {e}"
        pos += step


@pytest.mark.parametrize("mix", ["q4_k_m", "q4_k"])
def test_prefill_of_many_tokens_with_4096_wide_rows(mix):
    """80 and 70 tokens a step at hidden = 4096: q|k(|v) as one product read through row strides, gate|up as
    one product over the paired matrix, SwiGLU applied by the down projection's activation preparation
    (Q4_K and, in the q4_k_m mix, Q6_K down projections on the int8 GEMM), then single-token steps."""
    cfg = dict(CFG, n_layer=2, hidden=4096, n_head=4, n_kv_head=2, head_dim=128, ffn=1024, vocab=512, n_ctx=192)
    m, o = make(cfg, 35, mix)
    rng = np.random.default_rng(15)
    toks = [int(t) for t in rng.integers(0, cfg["vocab"], size=153)]
    pos = 0
    for step in (80, 70, 1, 1, 1):
        chunk = toks[pos:pos + step]
        ok, e = close(m.forward(chunk, pos), o.forward(chunk, pos))
        assert ok, f"pos {pos} +{step}: {e}"
        pos += step


@pytest.mark.parametrize("n_head,n_kv", [(4, 1), (4, 2), (2, 2), (8, 1)])
def test_long_prefill_chunks(n_head, n_kv):
    """Attention on split f16 operands with four, two, one and eight query heads a KV head: a chunk from position 0, chunks
    that start inside a key tile, an odd number of key tiles, a last tile part empty."""
    cfg = dict(CFG, n_ctx=400, n_layer=2, head_dim=128, n_head=n_head, n_kv_head=n_kv)
    m, o = make(cfg, 33)
    rng = np.random.default_rng(14)
    toks = [int(t) for t in rng.integers(0, cfg["vocab"], size=390)]
    pos = 0
    for step in (137, 150, 9, 94):
        chunk = toks[pos:pos + step]
        ok, e = close(m.forward(chunk, pos), o.forward(chunk, pos))
        assert ok, f"pos {pos} +{step}: {e}"
        pos += step


@pytest.mark.parametrize("n_head,n_kv", [(4, 1), (4, 2), (2, 2), (8, 1)])
def test_short_prefill_chunks(n_head, n_kv):
    """Steps of 9 to 31 tokens below 128 keys, on the f32 matrix cores with the same head counts: whole and part tiles of 16
    tokens and keys, up to the line from which the split operands take over and one step past it."""
    cfg = dict(CFG, n_ctx=160, n_layer=2, head_dim=128, n_head=n_head, n_kv_head=n_kv)
    m, o = make(cfg, 34)
    toks = [int(t) for t in np.random.default_rng(16).integers(0, cfg["vocab"], size=160)]
    pos = 0
    for step in (9, 16, 31, 17, 24, 30, 20):
        chunk = toks[pos:pos + step]
        ok, e = close(m.forward(chunk, pos), o.forward(chunk, pos))
        assert ok, f"pos {pos} +{step}: {e}"
        pos += step


@pytest.mark.parametrize("n_head,n_kv,steps", [(8, 2, (32, 31, 64, 9, 8, 96)), (8, 2, (63, 64, 9)), (8, 2, (64, 63, 9)),
                                                (8, 8, (129, 33)), (16, 1, (160, 40)), (24, 2, (32, 31, 40)), (12, 6, (127, 128, 1)), (20, 4, (40, 60))])
def test_attention_of_many_tokens_over_values_of_different_size(n_head, n_kv, steps):
    """Steps on both sides of the line from which attention runs on split f16 operands (64 tokens, or 128 keys; with 12 and 16
    heads a KV head 32 tokens), with 4, 1, 16, 12, 2 and 5 query heads a KV head (the last on the general kernel), part tiles of keys and tokens.  Every third token's
    values are some 200 times the others', and the first 40 tokens hold none of those: the value tiles' scales differ."""
    cfg = dict(CFG, n_ctx=256, n_layer=2, head_dim=128, n_head=n_head, n_kv_head=n_kv, hidden=256, vocab=600)
    rng = np.random.default_rng(n_head)
    wide = rng.normal(size=(600, 256)) * np.where(np.arange(256) < 32, 1e-3, 1.0)
    wide[400:, :32] = rng.normal(size=(200, 32)) * 3.0                   # tokens 400 .. carry the first 32 columns
    over = {"token_embd.weight": (capi.Q8_0, synth.quantize(capi.Q8_0, wide.astype(np.float32)))}
    for i in range(2):
        v = rng.normal(size=(n_kv * 128, 256)) / 16.0 * np.where(np.arange(256) < 32, 100.0, 0.5)
        over[f"blk.{i}.attn_v.weight"] = (capi.Q8_0, synth.quantize(capi.Q8_0, v.astype(np.float32)))
    m, o = make(cfg, 51, override=over)
    pos = 0
    for n in steps:
        t = np.arange(pos, pos + n)
        toks = np.where((t >= 40) & (t % 3 == 0), rng.integers(400, 600, size=n), rng.integers(0, 400, size=n))
        ok, e = close(m.forward(toks, pos), o.forward([int(x) for x in toks], pos))
        assert ok, f"pos {pos} +{n}: {e}"
        pos += n


@pytest.mark.parametrize("by", [112, -104])
def test_attention_of_many_tokens_over_values_at_the_ends_of_f32(by):
    """MXFP4 values 2^by times an ordinary model's behind an output projection of 2^-by: the same logits."""
    cfg = dict(CFG, n_ctx=256, n_layer=2, head_dim=128, n_head=8, n_kv_head=2, hidden=256)
    logits = []
    for b in (0, by):
        over = {}
        for i in range(2):
            for name, n, k, e in (("attn_v", 256, 256, b), ("attn_output", 256, 1024, -b)):
                raw = np.array(synth.normal_quantized(capi.MXFP4, 70 + i, n * k, 1.0)).view(np.uint8).reshape(-1, 17)
                raw[:, 0] = raw[:, 0].astype(np.int64) + e
                over[f"blk.{i}.{name}.weight"] = (capi.MXFP4, raw.reshape(-1))
        m, _ = make(cfg, 52, override=over)
        logits.append(np.stack([m.forward(list(range(100, 230)), 0), m.forward(list(range(300, 340)), 130)]))
    ok, e = close(logits[1], logits[0])
    assert ok, e


def test_attention_of_many_tokens_holds_every_operand_to_more_than_f16():
    """One layer over 200 tokens against 64 bits.  The embeddings are unit vectors, so that queries, keys and values are columns
    of their weights, and the down projection is zero: the error is the attention's and that of the 16-bit activations of the
    two products behind it (half a step of 2^-15 of the largest of 256 each).  An operand that was held to f16 alone would
    show: each is rounded in turn here, on the CPU, and is twice over the bound or more."""
    nh, nkv, h, S, rng = 8, 2, 256, 200, np.random.default_rng(8)
    cfg = dict(CFG, n_ctx=256, n_layer=1, hidden=h, head_dim=128, n_head=nh, n_kv_head=nkv, ffn=256, vocab=256)
    q8 = lambda v: (capi.Q8_0, synth.quantize(capi.Q8_0, np.ascontiguousarray(v, dtype=np.float32)))
    over = {"token_embd.weight": q8(np.eye(256)), "output.weight": q8(rng.normal(size=(256, h))),
            "blk.0.ffn_down.weight": q8(np.zeros((h, 256))), "blk.0.attn_output.weight": q8(rng.normal(size=(h, nh * 128)) * 0.2),
            "blk.0.attn_q_norm.weight": (0, (3.0 + rng.normal(size=128)).astype(np.float32))}
    over.update({f"blk.0.attn_{n}.weight": q8(rng.normal(size=(r * 128, h))) for n, r in (("q", nh), ("k", nkv), ("v", nkv))})
    m, o = make(cfg, 55, override=over)
    W = {n: oracle.dequantize(t, d).reshape(-1, nh * 128 if n == "blk.0.attn_output.weight" else 256).astype(np.float64)
         for n, (t, d) in o.t.items() if t != 0}
    F = {n: np.asarray(d).astype(np.float64) for n, (t, d) in o.t.items() if t == 0}
    toks = rng.permutation(256)[:S]
    got = m.logits_at(toks, 0, list(range(S)))

    rms = lambda v, w: v / np.sqrt((v * v).mean(-1, keepdims=True) + cfg["rms_eps"]) * w
    angle = np.arange(S)[:, None, None] * cfg["rope_theta"] ** (-np.arange(64) / 64.0)
    turn = lambda v: np.concatenate([v[..., :64] * np.cos(angle) - v[..., 64:] * np.sin(angle),
                                     v[..., 64:] * np.cos(angle) + v[..., :64] * np.sin(angle)], -1)
    x = W["token_embd.weight"][toks]
    n1 = rms(x, F["blk.0.attn_norm.weight"])
    q, k, v = ((n1 @ W[f"blk.0.attn_{n}.weight"].T).reshape(S, -1, 128) for n in "qkv")
    q, k = turn(rms(q, F["blk.0.attn_q_norm.weight"])), turn(rms(k, F["blk.0.attn_k_norm.weight"]))

    def logits(**rounded):
        r = {n: rounded.get(n, lambda v: v) for n in ("queries", "keys", "values", "weights")}
        ctx = []
        for i in range(nh):
            s = r["queries"](q[:, i]) @ r["keys"](k[:, i // 4]).T
            s = np.where(np.tri(S, dtype=bool), s / np.sqrt(128.0), -np.inf)
            e = np.exp(s - s.max(1, keepdims=True))
            ctx.append(r["weights"](e) @ r["values"](v[:, i // 4]) / e.sum(1, keepdims=True))
        return rms(x + np.concatenate(ctx, 1) @ W["blk.0.attn_output.weight"].T, F["output_norm.weight"]) @ W["output.weight"].T

    want = logits()
    err = lambda y: np.linalg.norm(y - want) / np.linalg.norm(want)
    f16 = lambda v: v.astype(np.float16).astype(np.float64)
    assert err(got) < 3e-5, err(got)
    for n in ("queries", "keys", "values", "weights"):
        assert err(logits(**{n: f16})) > 8e-5, (n, err(logits(**{n: f16})))


@pytest.mark.parametrize("at", [0, 45, 79])
def test_a_token_that_is_not_finite_stays_out_of_those_in_front(at):
    """Steps of 80 and 48 tokens, whose attention takes keys in tiles of 32: a token whose embedding is NaN is in the logits of
    those behind it and in none in front."""
    cfg = dict(CFG, n_ctx=160, n_layer=2, head_dim=128, n_head=8, n_kv_head=2)
    emb = np.random.default_rng(4).normal(size=(768, 512)).astype(np.float32)
    blocks = synth.quantize(capi.Q8_0, emb).copy()
    np.asarray(blocks).view(np.uint8).reshape(768, -1)[700, :2] = (0x00, 0x7E)   # the scale of its first block: NaN
    m, o = make(cfg, 53, override={"token_embd.weight": (capi.Q8_0, blocks)})
    toks = [int(t) for t in np.random.default_rng(5).integers(0, 700, size=128)]
    front = [p for p in range(0, 80, 3) if p < at] + ([at - 1] if at else [])
    behind = [p for p in (at, 46, 64, 79) if p >= at]
    ref = [o.forward(toks[:p + 1], 0) for p in front[-1:]]
    toks[at] = 700
    m.reset()
    got = m.logits_at(toks[:80], 0, front + behind)
    assert np.isfinite(got[:len(front)]).all() and not np.isfinite(got[len(front):]).any()
    if front:
        ok, e = close(got[len(front) - 1], ref[0])
        assert ok, e
    assert not np.isfinite(m.logits_at(toks[80:], 80, [0, 47])).any()


@pytest.mark.parametrize("head_dim,n_head,n_kv", [(64, 4, 2), (128, 4, 1), (256, 2, 2), (192, 4, 2), (128, 8, 1),
                                                  (128, 2, 2), (128, 4, 2)])
def test_decode_over_several_key_chunks(head_dim, n_head, n_kv):
    """A cache longer than one 64-key chunk of the split attention kernel, entered both by a
    long prefill and by short multi-token steps; head sizes with and without a split kernel.  The
    multi-token steps with head size 128 run the tiled matrix-core attention, with 8, 4, 2 and 1 query
    heads a KV head, token counts that do not fill a tile and keys already in the cache."""
    cfg = dict(CFG, n_ctx=224, n_layer=2, head_dim=head_dim, n_head=n_head, n_kv_head=n_kv)
    m, o = make(cfg, 26)
    rng = np.random.default_rng(3)
    toks = [int(t) for t in rng.integers(0, cfg["vocab"], size=190)]
    ok, e = close(m.forward(toks[:150], 0), o.forward(toks[:150], 0))
    assert ok, f"prefill: {e}"
    pos = 150
    for step in (1, 5, 8, 1, 3, 1, 1):
        chunk = toks[pos:pos + step]
        ok, e = close(m.forward(chunk, pos), o.forward(chunk, pos))
        assert ok, f"pos {pos} +{step}: {e}"
        pos += step


def test_replacing_a_tensor_after_decoding_takes_effect():
    """Single-token steps run q|k|v and gate|up as fused launches; a tensor set afterwards must win."""
    tensors = {n: (qt, d) for n, qt, d in qwen3_tensors(CFG, 27)}
    m, o = make(CFG, 27)
    m.forward([5, 6, 7], 0)
    m.forward([8], 3)                       # builds the fused copies
    other = {n: (qt, d) for n, qt, d in qwen3_tensors(CFG, 28)}
    for name in ("blk.1.attn_k.weight", "blk.2.ffn_up.weight"):
        tensors[name] = other[name]
        m.set_tensor(name, *other[name])
    o2 = oq.Qwen3Oracle(CFG, tensors, avx2=oracle.have_avx2())
    m.reset()
    ref = o2.forward([5, 6, 7], 0)
    ok, e = close(m.forward([5, 6, 7], 0), ref)
    assert ok, e
    ok, e = close(m.forward([8], 3), o2.forward([8], 3))
    assert ok, e


def test_position_contract_and_reset():
    m, _ = make(CFG, 23)
    a = m.forward([1, 2, 3], 0)
    with pytest.raises(capi.JoshuaHipError, match="does not match"):
        m.forward([4], 5)
    with pytest.raises(capi.JoshuaHipError, match="exceed the context"):
        m.forward(list(range(46)), 3)
    with pytest.raises(capi.JoshuaHipError, match="out of range"):
        m.forward([768], 3)
    with pytest.raises(capi.JoshuaHipError, match="at least one token"):
        m.forward([], 3)
    m.reset()
    b = m.forward([1, 2, 3], 0)
    assert np.array_equal(a, b)


def test_missing_tensor_is_reported():
    c = capi.Qwen3Config(1, 256, 2, 1, 64, 256, 256, 8, 1e-6, 1e4)
    m = capi.Qwen3(c)
    with pytest.raises(capi.JoshuaHipError, match="missing tensor"):
        m.forward([1], 0)
    with pytest.raises(capi.JoshuaHipError, match="unknown tensor"):
        m.set_tensor("blk.0.nope.weight", 0, np.zeros(4, np.float32))
    with pytest.raises(capi.JoshuaHipError, match="expected"):
        m.set_tensor("output_norm.weight", 0, np.zeros(4, np.float32))


def test_greedy_returns_last_index_of_equal_logits():
    # every row of the head identical -> all logits equal -> the last index wins
    from joshua_amd.synth import normal, quantize
    row = normal(5, (1, CFG["hidden"]), 0.05)
    head = quantize(8, np.repeat(row, CFG["vocab"], axis=0))
    m, _ = make(CFG, 24, override={"output.weight": (8, head)})
    logits = m.forward([1, 2], 0)
    assert np.all(logits == logits[0])
    assert m.greedy() == CFG["vocab"] - 1


def test_tied_embeddings_when_no_output_head():
    tensors = {n: (qt, d) for n, qt, d in qwen3_tensors(CFG, 25)}
    del tensors["output.weight"]
    c = capi.Qwen3Config(CFG["n_layer"], CFG["hidden"], CFG["n_head"], CFG["n_kv_head"], CFG["head_dim"], CFG["ffn"],
                         CFG["vocab"], CFG["n_ctx"], CFG["rms_eps"], CFG["rope_theta"])
    m = capi.Qwen3(c)
    for n, (qt, d) in tensors.items():
        m.set_tensor(n, qt, d)
    o = oq.Qwen3Oracle(CFG, tensors, avx2=oracle.have_avx2())
    ok, e = close(m.forward([9, 8, 7], 0), o.forward([9, 8, 7], 0))
    assert ok, e


FALLBACK_CHILD = r"""
import sys, numpy as np
sys.path.insert(0, %r)
from tests.test_gpu_qwen3 import CFG, make, close
cfg = dict(CFG, n_layer=2, hidden=4096, n_head=4, n_kv_head=2, head_dim=128, ffn=512, vocab=512, n_ctx=32)
m, o = make(cfg, 33, "q4_k")
pos = 0
for chunk in ([3, 500, 41], [7], [9], [256, 12]):
    ok, e = close(m.forward(chunk, pos), o.forward(chunk, pos))
    assert ok, (pos, e)
    pos += len(chunk)
print("fallback ok")
"""


@pytest.mark.parametrize("env", [{"JQ_Q4K_DOT4": "0"}, {"JQ_NO_FUSED_NORM": "1"}, {"JQ_NO_PAIRED_GATE_UP": "1"}])
def test_single_token_steps_without_the_fused_launches(env):
    """The switches are read when the library first dispatches, so each runs in a child process: without
    the v_dot4 kernel the row-paired gate|up matrix goes through the plain product and a pairwise
    SwiGLU; without the fused norm the pieces run as launches of their own; without pairing gate and up
    are laid one after the other."""
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    res = subprocess.run([sys.executable, "-c", FALLBACK_CHILD % root], env=dict(os.environ, **env), capture_output=True,
                         text=True, timeout=110)
    assert res.returncode == 0 and "fallback ok" in res.stdout, res.stdout + res.stderr


def test_short_step_across_a_key_chunk_boundary_after_a_longer_context():
    """A step of 2..8 tokens whose first tokens end before a 64-key chunk that its last tokens reach:
    those tokens have no sums for that chunk, and the buffer of partial sums still holds an earlier,
    longer context's values (laid out for more chunks, so its -inf markers sit where sums are read now).
    The merge must leave such chunks out; weighting them by zero turns inf into NaN."""
    cfg = dict(CFG, n_ctx=224, n_layer=2)
    m, o = make(cfg, 35)
    rng = np.random.default_rng(6)
    toks = [int(t) for t in rng.integers(0, cfg["vocab"], size=200)]
    m.forward(toks[:124], 0)
    m.forward(toks[124:132], 124)           # 3 chunks; tokens 0..3 stop at key 127 and skip the third
    m.forward(toks[132:196], 132)
    m.forward(toks[196:198], 196)           # 4 chunks: 196 keys for token 0 ... stride of the buffer changes
    m.reset()
    got, ref = m.forward(toks[:60], 0), o.forward(toks[:60], 0)
    ok, e = close(got, ref)
    assert ok, f"prefill: {e}"
    for pos, step in ((60, 8), (68, 1), (69, 3)):     # 60 + 8 crosses key 64; tokens 0..3 skip chunk 1
        chunk = toks[pos:pos + step]
        got, ref = m.forward(chunk, pos), o.forward(chunk, pos)
        assert np.all(np.isfinite(got)), f"pos {pos} +{step}: non-finite logits"
        ok, e = close(got, ref)
        assert ok, f"pos {pos} +{step}: {e}"


def test_long_context_with_five_query_heads_a_kv_head():
    """5 query heads a KV head take the one-row-per-workgroup attention for steps of more than 8 tokens;
    its scores go by in chunks, so a context of more than 16384 keys (64 KB of scores a row) works.
    Prefill in chunks of 2048 up to 16384 tokens, then a 16-token step whose rows see up to 16400 keys."""
    cfg = dict(n_layer=1, hidden=256, n_head=5, n_kv_head=1, head_dim=64, ffn=256, vocab=256, n_ctx=16400 + 16,
               rms_eps=1e-6, rope_theta=1e6)
    m, o = make(cfg, 36, "8")            # Q8_0: blocks of 32 fit the 320-wide attention output
    rng = np.random.default_rng(7)
    toks = [int(t) for t in rng.integers(0, cfg["vocab"], size=16400)]
    pos = 0
    while pos < 16384:
        m.forward_only(toks[pos:pos + 2048], pos)
        o.forward(toks[pos:pos + 2048], pos)
        pos += 2048
    got, ref = m.forward(toks[pos:pos + 16], pos), o.forward(toks[pos:pos + 16], pos)
    ok, e = close(got, ref)
    assert ok, e


def test_logits_in_host_memory_are_those_on_the_device():
    """One row, three rows (odd counts of floats) and 40, which are more than what leaves through pinned memory at once."""
    import torch
    from joshua_amd.capi import lib
    m, _ = make(dict(CFG, n_layer=1, vocab=30001, n_ctx=64), 91, "q4_k")
    t = np.random.default_rng(3).integers(0, 30001, 40).astype(np.uint32)
    for want in ([39], [0, 17, 39], list(range(40)), [39]):
        w = np.array(want, np.uint32)
        host, dev = np.full((w.size, 30001), np.nan, np.float32), torch.full((w.size, 30001), float("nan"), device="cuda")
        for ptr, on_device in ((host.ctypes.data, 0), (dev.data_ptr(), 1)):
            m.reset()
            assert lib().jq_model_forward(m._h, t.ctypes.data, t.size, 0, w.ctypes.data, w.size, ptr, on_device, None) == 0
        torch.cuda.synchronize()
        assert np.isfinite(host).all() and np.array_equal(host, dev.cpu().numpy()), want


@pytest.mark.parametrize("n_head,n_kv,d", [(64, 8, 64), (32, 4, 128), (16, 16, 256)])
def test_output_projection_that_merges_the_attention_of_a_step(n_head, n_kv, d):
    """Attention results of 4096 values into a Q4_K output projection: one to eight chunks of 64 keys are merged in the product's
    start (up to four, and up to eight), nine by a launch of their own."""
    cfg = dict(CFG, n_layer=1, hidden=2048, n_head=n_head, n_kv_head=n_kv, head_dim=d, ffn=256, vocab=512, n_ctx=520)
    m, o = make(cfg, 95, "q4_k")
    toks = np.random.default_rng(16).integers(0, 512, 520).tolist()
    pos = 0
    for prompt, steps in ((3, 2), (57, 4), (120, 6), (65, 3), (190, 4), (55, 6)):
        for n in [prompt] + [1] * steps:
            ok, e = close(m.forward(toks[pos:pos + n], pos), o.forward(toks[pos:pos + n], pos))
            assert ok, f"pos {pos}: {e}"
            pos += n
    assert pos > 512


MERGE_CHILD = r"""
import sys, numpy as np
sys.path.insert(0, sys.argv[1])
from tests.test_gpu_qwen3 import CFG, make
out = []
for n_head, n_kv, d in ((64, 8, 64), (32, 4, 128)):
    m, _ = make(dict(CFG, n_layer=1, hidden=2048, n_head=n_head, n_kv_head=n_kv, head_dim=d, ffn=256, vocab=512, n_ctx=520), 96, "q4_k")
    toks, pos = np.random.default_rng(18).integers(0, 512, 520).tolist(), 0
    for prompt in (3, 60, 70, 130, 200):
        m.forward(toks[pos:pos + prompt], pos)
        pos += prompt
        for _ in range(3):
            out.append(m.forward(toks[pos:pos + 1], pos))
            pos += 1
np.save(sys.argv[2], np.stack(out))
"""


def test_merging_in_the_output_projection_leaves_the_bits_of_the_merging_launch(tmp_path):
    import os
    import subprocess
    import sys
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    got = []
    for name, env in (("merged", {}), ("apart", {"JQ_NO_MERGE_IN_GEMV": "1"})):
        path = str(tmp_path / (name + ".npy"))
        res = subprocess.run([sys.executable, "-c", MERGE_CHILD, root, path], env=dict(os.environ, **env), capture_output=True, text=True,
                             timeout=110)
        assert res.returncode == 0, res.stdout + res.stderr
        got.append(np.load(path))
    assert np.isfinite(got[0]).all() and np.array_equal(got[0].view(np.uint32), got[1].view(np.uint32))


@pytest.mark.parametrize("mix", ["q4_k_m", "q4_k"])
def test_single_token_steps_with_1536_wide_rows(mix):
    """hidden = 1536: residual add, RMSNorm and product of a single token as one launch of six waves a tile, the stored residual row and
    (q4_k_m: an attn_v of another format) the stored normalised row among its results."""
    cfg = dict(CFG, n_layer=4, hidden=1536, n_head=4, n_kv_head=2, head_dim=128, ffn=768, vocab=512, n_ctx=40)
    m, o = make(cfg, 37, mix)
    if mix == "q4_k_m":
        assert any(qt != capi.Q4_K for n, qt, _ in qwen3_tensors(cfg, 37, mix) if n.endswith("attn_v.weight"))
    toks, pos = np.random.default_rng(19).integers(0, 512, 24).tolist(), 0
    for n in (5, 1, 1, 1, 9, 1, 1):
        ok, e = close(m.forward(toks[pos:pos + n], pos), o.forward(toks[pos:pos + n], pos))
        assert ok, f"pos {pos}: {e}"
        pos += n


@pytest.mark.parametrize("ffn,tokens", [(2048, 128), (2304, 131), (2304, 257), (3840, 160)])
def test_gate_and_up_of_many_tokens(ffn, tokens):
    """hidden = 1024: gate and up as products of their own, SwiGLU between two launches; a down projection of Q4_K and of Q6_K."""
    cfg = dict(CFG, n_layer=4, hidden=1024, n_head=8, n_kv_head=2, head_dim=128, ffn=ffn, vocab=512, n_ctx=300)
    m, o = make(cfg, 41, "q4_k_m")
    toks = np.random.default_rng(23).integers(0, 512, tokens + 1).tolist()
    ok, e = close(m.forward(toks[:tokens], 0), o.forward(toks[:tokens], 0))
    assert ok, e
    ok, e = close(m.forward(toks[tokens:], tokens), o.forward(toks[tokens:], tokens))
    assert ok, e


@pytest.mark.parametrize("ffn,tokens,inside", [(4864, 257, True), (6144, 257, True), (8192, 257, True), (4096, 600, True), (2048, 131, False)])
def test_gate_and_up_of_many_tokens_with_the_activation_in_the_product(ffn, tokens, inside):
    """hidden = 4096 pairs gate and up rows.  SwiGLU where their product is stored, in workgroups of four waves and of eight with six, eight and
    seven groups of weight rows, rows ragged (and columns, of six and seven groups); in four parts of k, in the down projection's preparation.
    Down projections of Q4_K and of Q6_K."""
    cfg = dict(CFG, n_layer=4, hidden=4096, n_head=4, n_kv_head=2, head_dim=128, ffn=ffn, vocab=512, n_ctx=640)
    assert {qt for n, qt, _, _ in qwen3_tensor_plan(cfg, "q4_k_m") if n.endswith("ffn_down.weight")} == {capi.Q4_K, capi.Q6_K}
    rc, out = swiglu_product(np.zeros(2 * ffn * 16 * 144, np.uint8), 2 * ffn, np.ones((tokens, 4096), np.float32))
    assert (rc == 0 and not out[:-1].any()) if inside else rc == -1
    m, o = make(cfg, 41, "q4_k_m")
    toks = np.random.default_rng(23).integers(0, 512, tokens + 1).tolist()
    ok, e = close(m.forward(toks[:tokens], 0), o.forward(toks[:tokens], 0))
    assert ok, e
    ok, e = close(m.forward(toks[tokens:], tokens), o.forward(toks[tokens:], tokens))
    assert ok, e


@pytest.mark.parametrize("vocab", [4088, 4104])
def test_the_last_norm_in_front_of_and_inside_the_head(vocab):
    """Rows of 4096 of Q6_K: 511 tiles of eight rows take the norm as a launch, 513 take it into the product; the last position of several,
    single tokens, and a norm that is not finite."""
    cfg = dict(CFG, n_layer=1, hidden=4096, n_head=4, n_kv_head=2, head_dim=128, ffn=512, vocab=vocab, n_ctx=32)
    m, o = make(cfg, 43, "q4_k_m")
    assert {n: qt for n, qt, _ in qwen3_tensors(cfg, 43, "q4_k_m")}["output.weight"] == capi.Q6_K
    toks, pos = np.random.default_rng(29).integers(0, vocab, 16).tolist(), 0
    for n in (5, 1, 1):
        ok, e = close(m.forward(toks[pos:pos + n], pos), o.forward(toks[pos:pos + n], pos))
        assert ok, f"pos {pos}: {e}"
        pos += n
    w = np.ones(4096, np.float32)
    w[77] = np.nan
    m.set_tensor("output_norm.weight", 0, w)
    assert np.isnan(m.forward(toks[pos:pos + 1], pos)).all()
