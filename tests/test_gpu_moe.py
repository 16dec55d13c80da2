"""GPU parity of the MoE layer (router, top-k, grouped expert matmuls, combine)
against the CPU oracle, through the C ABI."""
import numpy as np
import pytest

import oracle
from oracle.moe import MoeOracle
from joshua_amd import capi, synth
from joshua_amd.synth import layered as sl

pytestmark = pytest.mark.gpu


def build(qtype, h, inter, E, k, seed, sigma=0.02, shared_inter=0, **kw):
    rw = synth.normal(seed, (E, h), sigma=0.02)
    gate = synth.normal_quantized(qtype, seed + 1, E * inter * h, sigma)
    up = synth.normal_quantized(qtype, seed + 2, E * inter * h, sigma)
    down = synth.normal_quantized(qtype, seed + 3, E * h * inter, sigma)
    shared_o = shared_w = None
    if shared_inter:
        sg = synth.normal_quantized(qtype, seed + 4, shared_inter * h, sigma)
        su = synth.normal_quantized(qtype, seed + 5, shared_inter * h, sigma)
        sd = synth.normal_quantized(qtype, seed + 6, h * shared_inter, sigma)
        shared_o = (qtype, shared_inter, sg, su, sd)
        shared_w = (capi.Weight.upload(qtype, sg, shared_inter, h), capi.Weight.upload(qtype, su, shared_inter, h),
                    capi.Weight.upload(qtype, sd, h, shared_inter))
    ora = MoeOracle(qtype, h, inter, E, k, rw, gate, up, down, shared=shared_o, avx2=oracle.have_avx2(), **kw)
    cfg = capi.MoeConfig(E, k, h, inter, 1 if kw.get("gating") == "sigmoid" else 0, 1 if kw.get("norm_topk", True) else 0,
                         float(kw.get("weights_scale", 0.0)), kw.get("n_group", 1), kw.get("topk_group", 1),
                         float(kw.get("swiglu_clamp", 0.0)), float(kw.get("swiglu_clamp_shared", 0.0)))
    dev = capi.Moe(cfg, rw, capi.Weight.upload(qtype, gate, E * inter, h), capi.Weight.upload(qtype, up, E * inter, h),
                   capi.Weight.upload(qtype, down, E * h, inter), router_bias=kw.get("router_bias"), shared=shared_w)
    return ora, dev


def close(got, want, tol=1e-3):
    return np.all(np.abs(got - want) <= tol * np.maximum(np.abs(want), 1.0))


@pytest.mark.parametrize("kw", [
    dict(), dict(norm_topk=False),
    dict(gating="sigmoid", weights_scale=2.5),
    dict(gating="sigmoid", n_group=4, topk_group=2, router_bias=np.linspace(-0.05, 0.05, 32).astype(np.float32)),
    dict(gating="softmax", n_group=8, topk_group=3),
])
def test_route_matches_oracle(kw):
    ora, dev = build(capi.Q8_0, 512, 32, 32, 6, 40, **kw)
    x = synth.normal(41, (9, 512))
    ids, w = dev.route(x)
    oid, ow = ora.route(x)
    assert np.array_equal(ids, oid)
    assert np.allclose(w, ow, rtol=2e-5, atol=1e-7)


@pytest.mark.parametrize("gating", ["sigmoid", "softmax"])
@pytest.mark.parametrize("E,groups,kept,used", [(256, 8, 4, 8), (256, 4, 1, 6), (96, 3, 2, 5), (40, 5, 2, 16), (24, 12, 7, 9), (60, 4, 2, 6)])
def test_route_of_experts_in_groups(gating, E, groups, kept, used):
    """Groups that lie in one slot of a wave's lanes (64, 32, 8 and 2 experts, the last slot part-filled), and 15, which do not; equal
    scores, and scores that are not numbers, go to the lower expert, each taken once."""
    bias = np.linspace(0.05, -0.05, E).astype(np.float32) if gating == "sigmoid" else None
    ora, dev = build(capi.Q8_0, 512, 32, E, used, 45 + E, gating=gating, n_group=groups, topk_group=kept, router_bias=bias)
    x = synth.normal(46, (11, 512))
    ids, w = dev.route(x)
    oid, ow = ora.route(x)
    assert np.array_equal(ids, oid)
    assert np.allclose(w, ow, rtol=2e-5, atol=1e-7)
    per = E // groups
    x[:] = 0.0
    x[1, 7], x[2, 500] = np.nan, np.inf
    ids, w = dev.route(x)
    if used <= kept * per:  # all scores equal, or falling with the expert's number
        assert np.array_equal(ids[0], np.arange(used)) and np.isfinite(w[0]).all()
    for row in ids:
        assert len(set(row.tolist())) == used and row.max() < E
    assert np.array_equal(ids[1], np.arange(used)) and np.isnan(w[1]).all()


@pytest.mark.parametrize("qtype,tokens", [(capi.Q4_K, 1), (capi.Q4_K, 2), (capi.Q4_K, 3), (capi.Q4_K, 9), (capi.BF16, 1), (capi.BF16, 4), (capi.BF16, 5), (capi.BF16, 8)])
def test_decode_sized_calls_over_experts_in_groups(qtype, tokens):
    """Gating inside the expert kernel up to 1024 workgroups of it (two tokens of Q4_K, four of plain rows), a launch of its own from there."""
    E, used, bias = (64, 8, 0.02) if qtype == capi.Q4_K else (16, 4, 0.02)
    kw = dict(gating="sigmoid", n_group=4, topk_group=2, weights_scale=2.5, router_bias=np.linspace(bias, -bias, E).astype(np.float32))
    x = synth.normal(47, (tokens, 512))
    if qtype == capi.Q4_K:
        ora, dev = build(qtype, 512, 512, E, used, 48, **kw)
        assert close(dev.forward(x), ora.forward(x))
        return
    inter, rw = 256, synth.normal(50, (E, 512), 0.05)
    w = [sl.to_bf16(synth.normal(51 + i, (E * n, k), k ** -0.5)) for i, (n, k) in enumerate([(inter, 512), (inter, 512), (512, inter)])]
    cfg = capi.MoeConfig(E, used, 512, inter, 1, 1, 2.5, 4, 2)
    dev = capi.Moe(cfg, rw, *(capi.Weight.upload(qtype, v, *v.shape) for v in w), router_bias=kw["router_bias"])
    gate, up, down = (sl.from_bf16(v).astype(np.float64).reshape(E, -1, v.shape[1]) for v in w)
    ids, wts = dev.route(x)
    logits = x.astype(np.float64) @ rw.astype(np.float64).T
    best = np.sort((1 / (1 + np.exp(-logits)) + kw["router_bias"]).reshape(tokens, 4, 4), 2)[:, :, 2:].sum(2).argsort(1)[:, 2:]
    assert all(set(row // 4) <= set(kept) for row, kept in zip(ids, best))
    want = np.zeros((tokens, 512))
    for t, v in enumerate(x.astype(np.float64)):
        for e, wt in zip(ids[t], wts[t]):
            g = gate[e] @ v
            want[t] += wt * (down[e] @ (g / (1 + np.exp(-g)) * (up[e] @ v)))
    # f32 sums of 512 and 256 terms: some 2^-24 of the terms' magnitudes a rounding
    assert np.abs(dev.forward(x) - want).max() <= 1e-5 * np.abs(want).max()


@pytest.mark.parametrize("h,E,tokens", [(544, 30, 45), (2080, 9, 33), (1024, 64, 128)])
def test_router_logits_of_many_tokens_are_those_of_few(h, E, tokens):
    """From 32 tokens on the logits come from a kernel that works on 8 experts x 8 tokens a workgroup (an expert
    count and a token count that are not multiples of 8, a row that ends inside a step of 1024 columns); it adds
    the same products in the same order, so ids and weights equal those of calls of 8 tokens bit for bit."""
    ora, dev = build(capi.Q8_0, h, 32, E, 4, 50 + E)
    x = synth.normal(51 + E, (tokens, h))
    ids, w = dev.route(x)
    assert np.array_equal(ids, ora.route(x)[0])
    for t0 in range(0, tokens, 8):
        i8, w8 = dev.route(x[t0:t0 + 8])
        assert np.array_equal(ids[t0:t0 + 8], i8) and np.array_equal(w[t0:t0 + 8], w8)


@pytest.mark.parametrize("tokens", [1, 2, 7, 64])
def test_qwen3moe_shaped_layer_q4k(tokens):
    """Qwen3-30B-A3B layer shape (h 2048, inter 768, top-8) with 16 experts."""
    ora, dev = build(capi.Q4_K, 2048, 768, 16, 8, 60)
    x = synth.normal(61 + tokens, (tokens, 2048))
    assert close(dev.forward(x), ora.forward(x))


def test_decode_and_grouped_dispatch_agree_on_device():
    """reference: src/quantized_qwen3_moe.rs:912-928 (prefill vs decode path, 1e-4)."""
    ora, dev = build(capi.Q4_K, 512, 256, 8, 2, 70)
    row = synth.normal(71, (1, 512))
    many = np.repeat(row, 9, axis=0)              # 18 pairs > 8 experts: grouped path
    one = dev.forward(row)
    assert np.all(np.abs(dev.forward(many) - one) < 1e-4)


@pytest.mark.parametrize("qtype", [capi.IQ2_XXS, capi.MXFP4, capi.Q6_K, capi.Q2_K, capi.Q8_0])
def test_deepseek_style_layer_with_shared_expert(qtype):
    ora, dev = build(qtype, 1024, 512, 16, 4, 80, shared_inter=512, gating="sigmoid", n_group=4, topk_group=2,
                     weights_scale=2.5, router_bias=np.linspace(-0.02, 0.02, 16).astype(np.float32))
    for tokens in (1, 5):
        x = synth.normal(81 + tokens, (tokens, 1024))
        assert close(dev.forward(x), ora.forward(x))


def test_shared_expert_of_another_width_runs_beside_the_groups():
    ora, dev = build(capi.Q4_K, 512, 512, 8, 2, 90, shared_inter=256, gating="sigmoid")
    for tokens in (1, 6):
        x = synth.normal(91 + tokens, (tokens, 512))
        assert close(dev.forward(x), ora.forward(x))


def test_q4k_groups_of_many_tokens_with_the_shared_expert_folded_in():
    """40 tokens: the shared expert's group holds all 40 (three passes of 16 in the grouped MFMA
    kernel), routed groups hold 0 to about 20."""
    ora, dev = build(capi.Q4_K, 1024, 768, 8, 2, 95, shared_inter=768, gating="sigmoid")
    x = synth.normal(96, (40, 1024))
    assert close(dev.forward(x), ora.forward(x))


@pytest.mark.parametrize("h,inter", [(4096, 256), (512, 2560), (256, 3072)])
def test_q4k_grouped_kernels_at_other_row_lengths(h, inter):
    """16-super-block gate/up rows (outside the fused MFMA kernel's reach), and down rows of 10 and
    12 super-blocks (two columns a wave)."""
    ora, dev = build(capi.Q4_K, h, inter, 4, 2, 97 + inter)
    x = synth.normal(98, (19, h))
    assert close(dev.forward(x), ora.forward(x))


@pytest.mark.parametrize("qtype,h,inter", [
    (capi.Q6_K, 768, 256),      # 630-byte rows: no aligned staging, plain kernels; 256-wide down rows: 16 lanes a row
    (capi.IQ2_XXS, 2560, 512),  # 660-byte rows: 4-byte staging
    (capi.IQ2_XXS, 1792, 256),  # 462-byte rows: plain kernels
    (capi.Q8_0, 96, 64),        # 102-byte rows, three blocks a row
    (capi.MXFP4, 160, 96),      # 85-byte rows
])
def test_row_lengths_that_change_the_staging(qtype, h, inter):
    ora, dev = build(qtype, h, inter, 8, 3, 100 + h)
    for tokens in (1, 11):
        x = synth.normal(101 + tokens, (tokens, h))
        assert close(dev.forward(x), ora.forward(x))


@pytest.mark.parametrize("tokens,E,k", [(300, 16, 4), (1000, 16, 4), (1024, 24, 4), (1100, 16, 4), (150, 160, 6),
                                        (500, 200, 8)])   # the last: a rank table of more than 64 KB
def test_many_tokens_are_grouped_by_expert_in_pair_order(tokens, E, k):
    """Pair lists of up to 4096 pairs are grouped by ranks within chunks of 64 pairs (one to four chunks a
    wave, a last chunk part empty, experts nobody picked); longer lists, or more chunks x experts than the
    LDS table holds, by one pass per expert.  A pair out of place would multiply a token by another expert
    or add it to another token's sum."""
    ora, dev = build(capi.Q8_0, 128, 64, E, k, 140 + tokens)
    x = synth.normal(141 + tokens, (tokens, 128))
    ids, _ = dev.route(x)
    assert np.array_equal(ids, ora.route(x)[0])
    assert close(dev.forward(x), ora.forward(x))


@pytest.mark.parametrize("qtype", [capi.Q4_K, capi.MXFP4, capi.IQ2_XXS])
def test_decode_sized_call_over_large_expert_matrices(qtype):
    """One token, expert matrices large enough that the integer-dot kernels take their activations
    from the separate quantisation launch rather than quantising them in every workgroup."""
    ora, dev = build(qtype, 2048, 4352, 2, 1, 120)
    x = synth.normal(121, (1, 2048))
    assert close(dev.forward(x), ora.forward(x))


@pytest.mark.parametrize("qtype,h,inter,E,k,shared_inter,tokens", [
    (capi.Q4_K, 2048, 768, 16, 4, 0, 4),          # 16 rows a workgroup, planes quantised by the workgroup
    (capi.MXFP4, 4096, 512, 16, 4, 512, 2),       # shared expert as a fifth pair
    (capi.IQ2_XXS, 4096, 2048, 8, 4, 2048, 1),    # planes copied from the quantisation launch, shared expert
    (capi.MXFP4, 4128, 2048, 8, 3, 0, 2),         # three pairs a token, two tokens
])
def test_decode_sized_down_projection_with_the_combine_fused(qtype, h, inter, E, k, shared_inter, tokens):
    """Decode-sized calls with 512 workgroups or more in the down projection: one launch walks each
    token's pairs and forms the weighted sum itself."""
    kw = dict(gating="sigmoid", weights_scale=2.5) if shared_inter else {}
    ora, dev = build(qtype, h, inter, E, k, 130 + h, shared_inter=shared_inter, **kw)
    x = synth.normal(131 + tokens, (tokens, h))
    want = ora.forward(x)
    assert close(dev.forward(x), want)
    assert close(dev.forward(x), want)


def test_many_tokens_group_beyond_the_lds_pair_list():
    ora, dev = build(capi.Q8_0, 64, 32, 4, 2, 110)
    x = synth.normal(111, (6200, 64))          # 12400 pairs
    ids, w = dev.route(x)
    oid, ow = ora.route(x)
    assert np.array_equal(ids, oid)
    assert close(dev.forward(x), ora.forward(x))


def test_moe_rejects_mismatched_shapes():
    gate = capi.Weight.upload(capi.Q8_0, synth.normal_quantized(capi.Q8_0, 1, 4 * 32 * 256, 0.02), 4 * 32, 256)
    down = capi.Weight.upload(capi.Q8_0, synth.normal_quantized(capi.Q8_0, 2, 4 * 256 * 32, 0.02), 4 * 256, 32)
    rw = synth.normal(3, (4, 256))
    with pytest.raises(capi.JoshuaHipError):
        capi.Moe(capi.MoeConfig(4, 5, 256, 32, 0, 1, 0.0, 1, 1), rw, gate, gate, down)      # k > E
    with pytest.raises(capi.JoshuaHipError):
        capi.Moe(capi.MoeConfig(4, 2, 256, 64, 0, 1, 0.0, 1, 1), rw, gate, gate, down)      # wrong inter


@pytest.mark.parametrize("qtype,h,inter,tokens,shared_inter", [
    (capi.Q4_K, 512, 256, 1, 0),       # decode-sized call, integer-dot kernel
    (capi.MXFP4, 512, 256, 2, 256),    # the same with a shared expert riding along as a group
    (capi.Q8_0, 512, 256, 1, 0),       # decode-sized call, f32 staged kernel
    (capi.Q4_K, 1024, 256, 40, 256),   # many tokens a group: the MFMA ring kernel, shared expert folded in
    (capi.Q6_K, 512, 256, 24, 0),      # many tokens a group, f32 staged kernel
    (capi.Q4_K, 512, 256, 3, 512),     # a shared expert of another width: launches of its own
])
def test_swiglu_clamp(qtype, h, inter, tokens, shared_inter):
    """Gate clamped from above and up on both sides before the activation, with a limit of its own for
    the shared expert (reference: src/quantized_deepseek4.rs:445-462, :2419-2448); limits low enough to bite."""
    kw = dict(swiglu_clamp=0.02, swiglu_clamp_shared=0.01)
    ora, dev = build(qtype, h, inter, 16, 4, 70, shared_inter=shared_inter, **kw)
    plain, _ = build(qtype, h, inter, 16, 4, 70, shared_inter=shared_inter)
    x = synth.normal(71, (tokens, h))
    want = ora.forward(x)
    assert not close(want, plain.forward(x))          # the limits change the result
    assert close(dev.forward(x), want)


@pytest.mark.parametrize("qtype,lead_blocks", [(capi.Q8_0, 1), (capi.MXFP4, 3), (capi.IQ2_XXS, 1), (capi.Q6_K, 1)])
def test_experts_that_are_views_at_odd_block_offsets(qtype, lead_blocks):
    """Expert stacks that start mid-buffer, a whole number of 34-, 17-, 66- or 210-byte blocks in: their
    first byte is 1- or 2-byte aligned while every row is a multiple of 4 bytes long, so the kernels that load
    rows into LDS four or sixteen bytes at a time must stand aside (one and five tokens: the decode-sized and
    the grouped dispatch)."""
    h, inter, E, k_used, seed = 1024, 512, 8, 2, 300 + qtype
    bb = oracle.block_geometry(qtype)[1]
    lead = lead_blocks * bb
    assert lead % 4 != 0
    parts, views = [], []
    for i, (rows, cols) in enumerate(((inter, h), (inter, h), (h, inter))):
        blocks = synth.normal_quantized(qtype, seed + i, E * rows * cols, 0.02)
        parts.append(blocks)
        buf = np.concatenate([np.zeros(lead, np.uint8), blocks])
        # the parent: one row of whole blocks that spans the buffer; the view: the stack behind the lead
        per_block = oracle.block_geometry(qtype)[0]
        parent = capi.Weight.upload(qtype, buf, 1, buf.size // bb * per_block)
        views.append(parent.view(lead, E * rows, cols))
    rw = synth.normal(seed + 9, (E, h), 0.02)
    ora = MoeOracle(qtype, h, inter, E, k_used, rw, parts[0], parts[1], parts[2], avx2=oracle.have_avx2())
    cfg = capi.MoeConfig(E, k_used, h, inter, 0, 1, 0.0, 1, 1, 0.0, 0.0)
    dev = capi.Moe(cfg, rw, views[0], views[1], views[2])
    for tokens in (1, 5):
        x = synth.normal(seed + 20 + tokens, (tokens, h))
        assert close(dev.forward(x), ora.forward(x)), (capi.TYPE_NAMES[qtype], tokens)
    dev.close()


@pytest.mark.parametrize("E,k,shared_inter", [(8, 7, 0), (8, 8, 256), (16, 14, 0)])
def test_one_token_that_takes_nearly_every_expert(E, k, shared_inter):
    """One token of Q4_K experts with short rows whose pairs hit most experts: by the estimate of costs it would be bucketed, but
    the kernels for one row a group take such a call to have a group a pair."""
    ora, dev = build(capi.Q4_K, 512, 256, E, k, 95 + E, shared_inter=shared_inter)
    for seed in range(3):
        x = synth.normal(96 + seed, (1, 512))
        assert close(dev.forward(x), ora.forward(x))


@pytest.mark.parametrize("tokens", [9, 20, 40])
def test_few_tokens_an_expert_take_the_int8_quads_kernel(tokens):
    """16 experts, top-2: 18 to 80 pairs over 16 experts is at most five a group on average, the range of the
    int8 kernel that multiplies four activation rows an MFMA (one quad, two quads, and groups of more than
    eight rows, which take a second pass over the weights); inter 768 gives its down projection three waves a
    workgroup, hidden 2048 its gate and up eight."""
    ora, dev = build(capi.Q4_K, 2048, 768, 16, 2, 90)
    x = synth.normal(91 + tokens, (tokens, 2048))
    if tokens == 40:
        x[:12] = x[0] + 0.01 * x[:12]                # a dozen tokens that route alike
    ids, _ = dev.route(x)
    counts = np.bincount(ids.reshape(-1), minlength=16)
    if tokens == 40:
        assert counts.max() > 8                      # at least one group needs two passes
    assert close(dev.forward(x), ora.forward(x))


@pytest.mark.parametrize("qtype,h,inter,E,k,tokens,shared_inter,kw,kernel", [
    (capi.Q4_K, 5120, 256, 8, 2, 40, 0, {}, "moe_gemm_i8_mixed"),    # rows too long for the Q4_K grouped kernels
    (capi.IQ2_XXS, 1024, 512, 8, 2, 70, 512, dict(gating="sigmoid", swiglu_clamp=0.02, swiglu_clamp_shared=0.01),
     "moe_gemm_i8_mixed"),                                           # the shared expert's 70 pairs: one tile of 128
    (capi.MXFP4, 512, 768, 16, 4, 33, 0, {}, "moe_gemm_i8_mixed"),
    (capi.Q6_K, 768, 256, 4, 2, 300, 0, {}, "moe_gemm_i8_mixed"),    # about 150 pairs an expert: a tile of 128 and one of 32
    (capi.Q2_K, 512, 256, 4, 2, 300, 0, dict(swiglu_clamp=0.02), "moe_gemm_i8_mixed"),
    (capi.Q8_0, 256, 512, 16, 4, 64, 512, dict(gating="sigmoid", weights_scale=2.5), "moe_gemm_i8_mixed"),
    (capi.MXFP4, 256, 256, 160, 6, 150, 0, {}, "moe_gemm_i8_few"),   # more experts than one pass of the tile plan; under 8 pairs an expert
    (capi.IQ2_XXS, 512, 512, 4, 2, 200, 0, {}, "moe_gemm_i8_mixed"),
    (capi.Q4_K, 512, 256, 4, 2, 300, 256, dict(gating="sigmoid"), "moe_gemm_i8_mixed"),  # 16 pairs an expert or more: ahead of the ring kernel
])
def test_many_tokens_take_the_grouped_int8_gemm(qtype, h, inter, E, k, tokens, shared_inter, kw, kernel):
    """Bucketed calls of the formats with a side of the int8 GEMM: pairs sorted by expert are laid out in row
    groups of 16 that never mix two experts, gate and up run from one preparation of the tokens, the activation
    is applied in place (with the shared expert's own clamp on its rows) and the down projection reads it.  Under 8
    pairs an expert on average: tiles of 32 rows whose waves share the weight rows; more: an expert's pairs in tiles of
    128 rows whose waves share the rows while 80 or more are left, the rest in tiles of 32 (two launches)."""
    ora, dev = build(qtype, h, inter, E, k, 150 + h, shared_inter=shared_inter, **kw)
    x = synth.normal(151 + tokens, (tokens, h))
    want = ora.forward(x)
    got = dev.forward(x)
    assert capi.last_kernel() == kernel
    assert close(got, want)
    assert np.array_equal(got, dev.forward(x))
    few = synth.normal(152, (3, h))                                   # then a decode-sized call on the same layer
    assert close(dev.forward(few), ora.forward(few))


@pytest.mark.parametrize("h,inter,E,k,tokens,shared_inter,kw", [
    (256, 256, 128, 4, 128, 0, {}),                                  # one super-block a row; 4 pairs an expert: tiles of one row group
    (768, 256, 130, 5, 260, 256, dict(gating="sigmoid", swiglu_clamp=0.02, swiglu_clamp_shared=0.01)),  # a folded shared expert of 260 rows: six tiles
    (512, 512, 64, 6, 400, 0, {}),                                   # 37 pairs an expert: two and three row groups
    (1024, 1024, 32, 8, 330, 0, dict(weights_scale=2.5)),            # 82 pairs an expert: a whole tile and a part
    (768, 768, 48, 4, 64, 768, {}),
])
def test_q4k_experts_on_split_f16_activations(h, inter, E, k, tokens, shared_inter, kw):
    """Four pairs an expert and more where the workgroups fill the chip: the products of Q4_K weights are exact and the activations
    held to 22 bits, so the layer lies within 1e-5 of the oracle's f32 (sums of 256 to 1024 f32 terms in another order)."""
    ora, dev = build(capi.Q4_K, h, inter, E, k, 500 + h + E, shared_inter=shared_inter, **kw)
    x = synth.normal(501 + tokens, (tokens, h)) * np.float32(4.0)
    x[:, :32] *= np.float32(1e-5)                                     # a sub-block far below its super-block
    got = dev.forward(x)
    assert capi.last_kernel() == "moe_split16"
    want = ora.forward(x)
    assert np.array_equal(got, dev.forward(x))
    assert np.abs(got - want).max() <= 1e-5 * max(1.0, np.abs(want).max())
    few = synth.normal(502, (3, h))                                   # then a decode-sized call on the same layer
    assert close(dev.forward(few), ora.forward(few))


@pytest.mark.parametrize("inter", [64, 96, 128])
def test_q4k_experts_of_few_columns_on_split_f16_activations(inter):
    """Up to 128 gate rows an expert (a down projection of another type: Q4_K has none so short): waves of two tiles."""
    h, E, k, T = 512, 256, 8, 140
    rw = synth.normal(670, (E, h), sigma=0.02)
    gate, up = (synth.normal_quantized(capi.Q4_K, 671 + i, E * inter * h, 0.02) for i in range(2))
    down = synth.normal_quantized(capi.Q8_0, 673, E * h * inter, 0.02)
    ora = MoeOracle(capi.Q4_K, h, inter, E, k, rw, gate, up, down, avx2=oracle.have_avx2(), qtype_down=capi.Q8_0)
    dev = capi.Moe(capi.MoeConfig(E, k, h, inter, 0, 1, 0.0, 1, 1, 0.0, 0.0), rw, capi.Weight.upload(capi.Q4_K, gate, E * inter, h),
                   capi.Weight.upload(capi.Q4_K, up, E * inter, h), capi.Weight.upload(capi.Q8_0, down, E * h, inter))
    x = synth.normal(674, (T, h)) * np.float32(20.0)
    got, want = dev.forward(x), ora.forward(x)
    assert capi.last_kernel() == "moe_split16" and close(got, want)


@pytest.mark.parametrize("alike", [0, 40])
def test_q4k_experts_on_split_f16_activations_against_64_bits(alike):
    """Ten pairs an expert, the calls that the ring kernel's f32 products ran before: no further from 64 bits than those.  The
    activations' 22 to 23 bits are 4e-8 of a product; the rest are the roundings of the f32 sums, fewer where the products with the
    low plane have sums of their own.  Norm of the error here: 5.9e-7, in one chain 7.3e-7; the ring kernel's, at 128
    experts of 2048 x 768, 6.3e-7."""
    h, inter, E, k, T = 2048, 512, 64, 8, 80
    ora, dev = build(capi.Q4_K, h, inter, E, k, 640)
    x = synth.normal(641, (T, h))
    x[:alike] = x[0] + np.float32(0.05) * x[:alike]                    # experts of 40 pairs and more beside others of a few
    got = dev.forward(x)
    assert capi.last_kernel() == "moe_split16"
    ids = np.asarray(dev.route(x)[0]).reshape(T, k)
    rows = [oracle.dequantize(capi.Q4_K, synth.normal_quantized(capi.Q4_K, 641 + i, E * inter * h, 0.02)).reshape(E, n, kk)
            for i, (n, kk) in enumerate(((inter, h), (inter, h), (h, inter)))]
    x = x.astype(np.float64)
    z = x @ synth.normal(640, (E, h), sigma=0.02).astype(np.float64).T
    want = np.zeros((T, h))
    top = np.take_along_axis(z, ids.astype(np.int64), 1)
    wts = np.exp(top - top.max(1, keepdims=True))
    wts /= wts.sum(1, keepdims=True)
    for e in range(E):
        t, slot = np.nonzero(ids == e)
        g, u, d = (r[e].astype(np.float64) for r in rows)
        a = x[t] @ g.T
        want[t] += wts[t, slot, None] * ((a / (1.0 + np.exp(-a)) * (x[t] @ u.T)) @ d.T)
    err = np.linalg.norm(got - want) / np.linalg.norm(want)
    assert err < 6.4e-7, err


def test_q4k_experts_on_split_f16_activations_near_the_end_of_f32():
    """Gated units of up to 1e36 or so are finite, and so is the layer, whose tokens are the powers of two apart that its results are."""
    h, inter, E, k, T = 512, 512, 64, 4, 300
    rw, x = synth.normal(660, (E, h), sigma=0.02), synth.normal(661, (T, h))
    w = [capi.Weight.upload(capi.Q4_K, synth.normal_quantized(capi.Q4_K, 662 + i, E * inter * h, 0.02), E * n, kk)
         for i, (n, kk) in enumerate(((inter, h), (inter, h), (h, inter)))]
    cfg = capi.MoeConfig(E, k, h, inter, 0, 1, 0.0, 1, 1, 0.0, 0.0)
    out = []
    for by in (2.0 ** 12, 2.0 ** 58):                                 # silu is max(., 0) but for gates of some 2^-8 of the rest
        out.append(capi.Moe(cfg, rw / np.float32(by), *w).forward(x * np.float32(by)).astype(np.float64) / by ** 2)
        assert capi.last_kernel() == "moe_split16"
    assert np.isfinite(out[1]).all()
    assert np.linalg.norm(out[1] - out[0]) <= 1e-5 * np.linalg.norm(out[0])


def test_q4k_experts_on_split_f16_activations_uneven_rows_and_non_finite_ones():
    """300 of 400 tokens route alike (experts with seven tiles, with one, and with none), one token holds a NaN and one an
    infinity: their rows come out NaN and nobody else's; the same layer with a down projection that the int8 GEMM runs."""
    ora, dev = build(capi.Q4_K, 512, 256, 128, 4, 611)
    x = synth.normal(612, (400, 512))
    x[:300] = x[0] + 0.01 * x[:300]
    x[7, 100], x[350, 300] = np.nan, np.inf
    got = dev.forward(x)
    assert capi.last_kernel() == "moe_split16"
    bad = np.zeros(400, bool)
    bad[[7, 350]] = True
    assert np.all(np.isnan(got[bad])) and np.all(np.isfinite(got[~bad]))
    want = ora.forward(x[~bad])
    ids, ref = dev.route(x[~bad])[0], ora.route(x[~bad])[0]
    same = np.array([set(a) == set(b) for a, b in zip(ids, ref)])     # (near-copies: a tie within rounding may fall otherwise)
    assert same.mean() > 0.95
    assert np.abs(got[~bad] - want)[same].max() <= 1e-5 * max(1.0, np.abs(want).max())
    ora, dev = build(capi.Q4_K, 256, 4096, 8, 2, 613)                 # 8 workgroups of 256 down rows
    x = synth.normal(614, (64, 256))
    assert close(dev.forward(x), ora.forward(x)) and capi.last_kernel() != "moe_split16"


@pytest.mark.parametrize("h,inter,E,k,tokens,shared_inter,kw", [
    (512, 512, 16, 4, 9, 0, {}),                                                  # one chunk a row; tiles of 8 pairs, most part-filled
    (1536, 512, 8, 2, 40, 512, dict(swiglu_clamp=0.02, swiglu_clamp_shared=0.01)),  # the shared expert's 40 pairs; limits that bite
    (1024, 2048, 4, 2, 100, 0, {}),                                               # 50 pairs an expert: tiles of 16 on eight waves in gate and up
    (4096, 1024, 32, 4, 130, 1024, dict(gating="sigmoid", weights_scale=2.5)),    # tiles of 16 in both, several column blocks a workgroup
    (512, 1536, 64, 8, 12, 0, {}),                                                # one or two pairs an expert
])
def test_mxfp4_experts_on_the_matrix_cores_fp4(h, inter, E, k, tokens, shared_inter, kw):
    """Bucketed MXFP4 calls on the FP4 matrix instructions: activations in 20 bits of their block's largest magnitude.
    Against a float64 layer over the exact weights, routed as the device routes: an activation is off by at most 2^-19 of its
    block's largest, in rms 2^-19 / sqrt 3 of it, and that largest is about 2.2 times the rms of a block of normal values, under
    6 times that of a block of products: 2.5e-6 through gate and as much through up, 7e-6 through down.  A row within 2^-16 = 1.5e-5
    of its norm (the 16-bit planes of the other kernels: 5e-5).  Gate values stay below about 0.1, twice the limits of the second
    case: beyond them most of a clamped sum cancels (this rounding alone, in float64, gives 4.7e-6 there and 1.5e-5 at 0.74)."""
    rw = synth.normal(900, (E, h), sigma=0.02)
    parts = [synth.normal_quantized(capi.MXFP4, 901 + i, E * inter * h, 0.02).copy() for i in range(3)]
    for p in parts:                       # the smallest scale, and blocks that stand for zeros (scale 0xFF)
        p.reshape(-1, 17)[::37, 0] = 0
        p.reshape(-1, 17)[5::41, 0] = 0xFF
    shp = [synth.normal_quantized(capi.MXFP4, 905 + i, shared_inter * h, 0.02) for i in range(3)] if shared_inter else []

    def up(b, n, kk):
        return capi.Weight.upload(capi.MXFP4, b, n, kk)

    shared = (up(shp[0], shared_inter, h), up(shp[1], shared_inter, h), up(shp[2], h, shared_inter)) if shp else None
    cfg = capi.MoeConfig(E, k, h, inter, int(kw.get("gating") == "sigmoid"), 1, kw.get("weights_scale", 0.0), 1, 1,
                         kw.get("swiglu_clamp", 0.0), kw.get("swiglu_clamp_shared", 0.0))
    dev = capi.Moe(cfg, rw, up(parts[0], E * inter, h), up(parts[1], E * inter, h), up(parts[2], E * h, inter), shared=shared)
    x = synth.normal(910 + tokens, (tokens, h)) * np.float32(2.0) ** (np.arange(tokens) % 9 - 12)[:, None].astype(np.float32)
    ids, wts = dev.route(x)
    got = dev.forward(x)
    assert capi.last_kernel() == "moe_mx"

    def deq(b, *shape):
        return oracle.dequantize(capi.MXFP4, b).reshape(shape).astype(np.float64)

    gw, uw, dw = deq(parts[0], E, inter, h), deq(parts[1], E, inter, h), deq(parts[2], E, h, inter)
    sh = [deq(shp[0], shared_inter, h), deq(shp[1], shared_inter, h), deq(shp[2], h, shared_inter)] if shp else None

    def ffn(v, a, b, c, limit):
        gt, upv = a @ v, b @ v
        if limit:
            gt, upv = np.minimum(gt, limit), np.clip(upv, -limit, limit)
        return c @ (gt / (1.0 + np.exp(-gt)) * upv)

    want = np.zeros((tokens, h))
    for t in range(tokens):
        v = x[t].astype(np.float64)
        for s in range(k):
            e = ids[t, s]
            want[t] += wts[t, s] * ffn(v, gw[e], uw[e], dw[e], kw.get("swiglu_clamp", 0.0))
        if shp:
            want[t] += ffn(v, *sh, kw.get("swiglu_clamp_shared", 0.0))
    rows = np.linalg.norm(got - want, axis=1) / np.linalg.norm(want, axis=1)
    assert rows.max() < 2.0 ** -16, rows.max()
    # rows that hold an inf or a NaN stay their own
    bad = x.copy()
    bad[1, 3], bad[tokens - 1, h - 1] = np.inf, np.nan
    again = dev.forward(bad)
    assert np.all(np.isnan(again[tokens - 1])) and not np.any(np.isfinite(again[1]))
    assert np.array_equal(again[[0] + list(range(2, tokens - 1))], got[[0] + list(range(2, tokens - 1))])


@pytest.mark.parametrize("tokens", [1, 3, 40, 200])
def test_tokens_that_are_not_finite_under_expert_groups(tokens):
    """Routing over groups of experts, on a layer that was never called: a token whose scores compare with nothing still gets
    experts (scratch holds none from before), its own row alone is NaN, and the others are what they are without it."""
    for seed in range(2):
        ora, dev = build(capi.Q4_K, 512, 256, 32, 6, 710 + seed, gating="sigmoid", n_group=4, topk_group=2, weights_scale=2.5,
                         router_bias=np.linspace(-0.05, 0.05, 32).astype(np.float32))
        x = synth.normal(711 + seed, (tokens, 512))
        bad = np.zeros(tokens, bool)
        bad[[0, tokens // 2, tokens - 1][:max(1, tokens // 3)]] = True
        x[bad, 17] = np.nan
        got = dev.forward(x)
        assert np.all(np.isnan(got[bad]))
        assert bad.all() or close(got[~bad], ora.forward(x[~bad]))
        ids, _ = dev.route(x)
        assert ids.max() < 32


@pytest.mark.parametrize("qtype", [capi.Q4_K, capi.MXFP4])
def test_grouped_int8_gemm_with_pairs_that_fall_unevenly(qtype):
    """260 of 300 tokens route alike: two experts get 260 pairs and more (two tiles of 128 and a tail of tiles of 32),
    the others a few each (tiles of 32 only), and experts without a pair get no tile."""
    ora, dev = build(qtype, 2048, 256, 16, 2, 171)
    x = 0.5 * synth.normal(172, (300, 2048))      # (the magnitude a normed layer gives: the GEMM's fixed point holds 1e-3 there)
    # a token whose second and third expert are well apart, so that its near-copies pick the same two
    logits = x[:40] @ ora.router_w.T
    top3 = np.sort(logits, axis=1)[:, -3:]
    x0 = x[int(np.argmax(top3[:, 1] - top3[:, 0]))].copy()
    x[:260] = x0 + 0.01 * x[:260]
    ids, _ = dev.route(x)
    assert np.array_equal(np.sort(ids, axis=1), np.sort(ora.route(x)[0], axis=1))
    counts = np.bincount(ids.reshape(-1), minlength=16)
    assert counts.max() >= 260 and counts.min() < 16
    got = dev.forward(x)
    assert capi.last_kernel() == "moe_gemm_i8_mixed"
    assert close(got, ora.forward(x))
    assert np.array_equal(got, dev.forward(x))


@pytest.mark.parametrize("qtype,h,inter,E,k,tokens,shared_inter,kw", [
    (capi.IQ2_XXS, 512, 512, 8, 2, 9, 0, {}),                       # 16 units a row: one a lane; 2 pairs an expert
    (capi.MXFP4, 1280, 384, 8, 3, 12, 384, {}),                     # 40 units over 16 lanes: a ragged third unit
    (capi.MXFP4, 4352, 128, 4, 2, 7, 128, dict(swiglu_clamp=0.5, swiglu_clamp_shared=0.25)),  # 136 units: 32 lanes, 5 a lane
    (capi.IQ2_XXS, 8704, 512, 4, 2, 5, 0, {}),                      # 272 units: 64 lanes, 5 a lane, rows of 2244 bytes
    (capi.IQ2_XXS, 1024, 4608, 6, 2, 40, 0, dict(gating="sigmoid")),  # down rows of 144 units; 13 pairs an expert
    (capi.MXFP4, 256, 2944, 5, 1, 30, 0, {}),                       # 2944 rows: 23 units (not a multiple of 4 x 16) in gate
    (capi.Q4_K, 512, 256, 8, 2, 9, 0, {}),                          # Q4_K: an offset a sub-block against the activations' sums
    (capi.Q4_K, 4096, 1536, 8, 2, 24, 1536, dict(swiglu_clamp=0.75, swiglu_clamp_shared=0.5)),  # Qwen3-235B-A22B row lengths
    (capi.Q4_K, 7168, 256, 4, 2, 6, 0, dict(gating="sigmoid")),     # rows of 28 super-blocks: seven units a lane
])
def test_few_pairs_an_expert_stream_past_weights_decoded_once(monkeypatch, qtype, h, inter, E, k, tokens, shared_inter, kw):
    """Bucketed calls of MXFP4, IQ2_XXS and Q4_K experts with few pairs an expert: moe_expert_dot8 keeps an expert's rows as
    int8 words in registers and streams the pairs' activation planes through LDS.  Row lengths that give one to
    eight units a lane on 16, 32 and 64 lanes a row, a last unit past the row's end, groups of one pair and of
    many, the folded shared expert (a group with a pair per token) and the clamped activation."""
    monkeypatch.setenv("JQ_MOE_EXPERT_DOT8_UPTO_PAIRS_PER_EXPERT", "1000")
    ora, dev = build(qtype, h, inter, E, k, 900 + h, shared_inter=shared_inter, **kw)
    x = synth.normal(901 + h, (tokens, h))
    got = dev.forward(x)
    assert capi.last_kernel() == "moe_expert_dot8"
    assert close(got, ora.forward(x))


def _random_expert_layers():
    rng = np.random.default_rng(20251125)
    cases = []
    for seed in range(10):
        qtype = [capi.MXFP4, capi.IQ2_XXS, capi.Q4_K][seed % 3]
        step = 512 if qtype == capi.IQ2_XXS else 256     # IQ2_XXS rows a multiple of 4 bytes: 512 columns
        for _ in range(100):
            h, inter = step * int(rng.integers(1, 17)), step * int(rng.integers(1, 7))
            E = int(rng.integers(2, 13))
            if h * inter * E <= 12 << 20:
                break
        k = int(rng.integers(1, min(E, 4) + 1))
        tokens = int(rng.integers(E // k + 1, 70))       # more pairs than experts
        shared = inter if rng.integers(0, 2) else 0
        cases.append((qtype, h, inter, E, k, tokens, shared, 950 + seed))
    return cases


@pytest.mark.parametrize("qtype,h,inter,E,k,tokens,shared_inter,seed", _random_expert_layers())
def test_expert_kernel_at_seeded_random_layers(monkeypatch, qtype, h, inter, E, k, tokens, shared_inter, seed):
    """moe_expert_dot8 at layer shapes drawn from a fixed seed: row lengths of 8 to 256 units (every lanes-a-row
    and units-a-lane combination comes up), 2 to 12 experts, top-1 to top-4, with and without the folded shared
    expert, against the oracle's layer.  The inputs are scaled so that gate and up results keep a standard
    deviation of about one at every row length, as a layer's normed activations give: unit-variance inputs
    against 8192 columns of weights of 0.02 make them 1.8 and the activations reach 50, where the fixed-point
    planes' error (in proportion to a row's largest magnitude) sits at the tolerance itself (one element of
    253952 at 1.06e-3)."""
    monkeypatch.setenv("JQ_MOE_EXPERT_DOT8_UPTO_PAIRS_PER_EXPERT", "1000")
    ora, dev = build(qtype, h, inter, E, k, seed, shared_inter=shared_inter)
    x = synth.normal(seed + 1, (tokens, h)) * np.float32(min(1.0, 1.0 / (0.02 * np.sqrt(h))))
    got = dev.forward(x)
    assert capi.last_kernel() == "moe_expert_dot8", (h, inter, E, k, tokens)
    assert close(got, ora.forward(x))


@pytest.mark.parametrize("tokens,shared", [(1, False), (3, False), (1, True)])
def test_q4k_experts_with_a_q6k_down_projection(tokens, shared):
    """The mix of a Q4_K_M file's layers with more bits: gate and up in Q4_K, down in Q6_K, rows of 768 (three
    210-byte blocks: 630 bytes, a multiple of neither 4 nor 16).  Decode-sized calls take the matrix-core kernels for
    both; the 16 rows of a down tile are copied as one span, which starts and ends on 16 bytes whatever the row."""
    h, inter, E, k = 2048, 768, 16, 4
    rw = synth.normal(700, (E, h), sigma=0.02)
    gate = synth.normal_quantized(capi.Q4_K, 701, E * inter * h, 0.02)
    up = synth.normal_quantized(capi.Q4_K, 702, E * inter * h, 0.02)
    down = synth.normal_quantized(capi.Q6_K, 703, E * h * inter, 0.02)
    sh_o = sh_w = None
    if shared:   # a shared expert of the same types and shape rides along as one more pair
        sg, su = (synth.normal_quantized(capi.Q4_K, 704 + i, inter * h, 0.02) for i in range(2))
        sd = synth.normal_quantized(capi.Q6_K, 706, h * inter, 0.02)
        sh_w = (capi.Weight.upload(capi.Q4_K, sg, inter, h), capi.Weight.upload(capi.Q4_K, su, inter, h),
                capi.Weight.upload(capi.Q6_K, sd, h, inter))
    ora = MoeOracle(capi.Q4_K, h, inter, E, k, rw, gate, up, down, avx2=oracle.have_avx2(), qtype_down=capi.Q6_K)
    cfg = capi.MoeConfig(E, k, h, inter, 0, 1, 0.0, 1, 1, 0.0, 0.0)
    dev = capi.Moe(cfg, rw, capi.Weight.upload(capi.Q4_K, gate, E * inter, h), capi.Weight.upload(capi.Q4_K, up, E * inter, h),
                   capi.Weight.upload(capi.Q6_K, down, E * h, inter), shared=sh_w)
    x = synth.normal(710 + tokens, (tokens, h))
    got = dev.forward(x)
    assert capi.last_kernel() == "moe_down_mfma"
    want = ora.forward(x)
    if shared:
        sx = np.ascontiguousarray(x, np.float32)
        g = oracle.matmul_t(capi.Q4_K, (tokens, h, inter), sx, sg, avx2=oracle.have_avx2())
        u = oracle.matmul_t(capi.Q4_K, (tokens, h, inter), sx, su, avx2=oracle.have_avx2())
        from oracle.moe import silu
        want = want + oracle.matmul_t(capi.Q6_K, (tokens, inter, h), (silu(g) * u).astype(np.float32), sd, avx2=oracle.have_avx2())
    assert close(got, want)
