"""Q4_K products of many activation rows on f16 and FP6 operands (kq_gemm_h6) against 64-bit products of the decoded weights.

The library takes the kernel from 128 activation rows on and picks the workgroup shape and the split over k by an estimate; with
both forced through the environment (read at the first dispatch, hence the child process) every shape runs at the edges of its
tiles."""
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle
from joshua_amd import capi, synth

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CHILD = r"""
import os, sys
import numpy as np
sys.path.insert(0, %r)
import oracle
from joshua_amd import capi, synth
splits = int(os.environ["JQ_GEMM_H6_SPLITS"])
name = "q4k_gemm_i8" + ("+splitk" if splits > 1 else "")


def parts(blocks, n, k):
    # p = sc (q - 8) of every element, its factor d, and the power of two in sc / 32 that its code stands on
    b = blocks.reshape(n, k // 256, 144)
    d = b[:, :, 0:2].copy().view(np.float16).astype(np.float64)[:, :, 0]
    s = b[:, :, 4:16].astype(np.int64)
    sc = np.concatenate([s[:, :, :4] & 63, (s[:, :, 8:] & 15) | s[:, :, :4] >> 6 << 4], 2)
    q = b[:, :, 16:].reshape(n, k // 256, 4, 1, 32)
    q = np.concatenate([q & 15, q >> 4], 3).reshape(n, k // 256, 8, 32).astype(np.int64)
    unit = 2.0 ** (np.floor(np.log2(np.maximum(sc, 1))) - 5)
    return (sc[..., None] * (q - 8)).astype(np.float64).reshape(n, -1, 256), d, unit.repeat(32, 2)


def check(blocks, lhs, what, rms=None):
    m, k = lhs.shape
    n = blocks.size // (k // 256 * 144)
    got = capi.Weight.upload(capi.Q4_K, blocks, n, k).matmul_t(m, lhs)
    assert (capi.last_kernel(), capi.last_arithmetic()) == (name, "f16+fp6"), (capi.last_kernel(), capi.last_arithmetic())
    w = oracle.dequantize(capi.Q4_K, blocks).reshape(n, k).astype(np.float64)
    x = lhs.astype(np.float64)
    want = x @ w.T
    # With s <= 2^-14 of a super-block's largest magnitude: the remainder l <= 8 s of an activation as E2M3 is at most s / 2 off,
    # p as E2M3 codes of 2^-7 p / unit at most max(|p| / 16, 8 unit): an element adds at most d s (|p| / 2 + 8 of that).  The mean of a
    # sub-block and its weight in two bf16 parts each: 2^-16 of the terms.  f32 sums: 2^-20 of them.
    p, d, unit = parts(blocks, n, k)
    s = np.abs(x.reshape(m, -1, 256)).max(2) * 2.0 ** -14
    off = np.abs(d) * (np.abs(p) / 2 + 8 * np.maximum(np.abs(p) / 16, 8 * unit)).sum(2)
    bound = s @ off.T + (2.0 ** -16 + 2.0 ** -20) * (np.abs(x) @ np.abs(w).T + np.abs(x) @ (np.abs(p) * np.abs(d)[..., None]).reshape(n, k).T)
    err = np.abs(got - want)
    assert np.all(err <= bound), (what, float((err / np.maximum(bound, 1e-300)).max()))
    if rms is not None:  # the remainders left out would show as 1e-4
        rel = np.sqrt((err ** 2).mean() / (want ** 2).mean())
        assert rel <= rms, (what, float(rel))
    return got


rng = np.random.default_rng(4)
sizes = [(17, 256, 64), (33, 512, 113), (64, 1024, 97), (129, 768, 112), (257, 512, 300), (256, 1024, 96)] if splits == 1 else [(40, 4096, 100), (300, 4096, 130)]
for m, k, n in sizes:
    check(synth.normal_quantized(capi.Q4_K, 5 + n, n * k, 0.02), synth.normal(6 + k, (m, k)), (m, k, n), 2e-5)
n, k = 80, 2048 if splits == 1 else 4096
raw = rng.integers(0, 256, (n * k // 256, 144), dtype=np.uint8)   # every scale, min and code
raw[:, 0:2] = (rng.uniform(-1e-3, 1e-3, n * k // 256)).astype(np.float16).view(np.uint8).reshape(-1, 2)
raw[:, 2:4] = (rng.uniform(-1e-3, 1e-3, n * k // 256)).astype(np.float16).view(np.uint8).reshape(-1, 2)
raw[::7, 0:2] = 0
lhs = synth.normal(9, (50, k))
check(raw.reshape(-1), lhs, "random blocks", 2e-5)
# rows whose groups of 16 span twelve orders of magnitude, of one non-zero element, with an empty stretch, at f32's ends
lhs[0] *= (10.0 ** rng.integers(-6, 7, size=k // 16)).repeat(16).astype(np.float32)
lhs[1] = 0
lhs[1, 1234] = 3.5
lhs[2, 512:1024] = 0
lhs[3] *= np.float32(1e30)
lhs[4] *= np.float32(1e-30)
lhs[5] = np.float32(65519.0)     # just below the next power of two's f16
got = check(raw.reshape(-1), lhs, "rows of every range")
lhs[7, 100], lhs[8, 2000], lhs[9, 5] = np.inf, np.nan, -np.inf
other = capi.Weight.upload(capi.Q4_K, raw.reshape(-1), n, k).matmul_t(50, lhs)
assert np.all(np.isnan(other[7:10])), "a row that is not finite"
assert np.array_equal(np.delete(other, [7, 8, 9], 0), np.delete(got, [7, 8, 9], 0)), "its neighbours"
# gate and up rows in turn: SwiGLU where the product is stored, in one part of k
from tests.h6_swiglu import swiglu_product
for m, k, n in [(17, 256, 64), (33, 512, 114), (64, 1024, 98), (129, 768, 112), (257, 512, 300), (256, 1024, 96), (40, 4096, 130)]:
    blocks, lhs = synth.normal_quantized(capi.Q4_K, 15 + n, n * k, 0.02), synth.normal(16 + k, (m, k))
    rc, got = swiglu_product(blocks, n, lhs)
    if splits > 1:
        assert rc == -1 and np.isnan(got).all()
        continue
    assert rc == 0 and np.isnan(got[m]).all() and np.isfinite(got[:m]).all(), (m, k, n)
    y = lhs.astype(np.float64) @ oracle.dequantize(capi.Q4_K, blocks).reshape(n, k).astype(np.float64).T
    gate, up = y[:, 0::2], y[:, 1::2]
    act = gate / (1 + np.exp(-gate))
    # the products are 2e-5 of their root mean square off (above) and silu's slope is at most 1.1; silu and the last product: some 2^-20
    rms = lambda v: np.sqrt((v ** 2).mean())
    assert rms(got[:m] - act * up) <= 2e-5 * rms(up) * (1.1 * rms(gate) + rms(act)) + 1e-6 * rms(act * up), (m, k, n)
    assert np.abs(got[:m] - act * up).max() <= 12 * 2e-5 * (1.1 * rms(gate) * np.abs(up).max() + np.abs(act).max() * rms(up)), (m, k, n)
assert swiglu_product(synth.normal_quantized(capi.Q4_K, 8, 113 * 512, 0.02), 113, synth.normal(9, (33, 512)))[0] == -1  # a gate without its up
# a decoder's prompt over such rows (4096 wide): in one part of k as above, in several the down projection's preparation applies SwiGLU
from tests.test_gpu_qwen3 import CFG, make, close
m, o = make(dict(CFG, n_layer=2, hidden=4096, n_head=4, n_kv_head=2, head_dim=128, ffn=4096, n_ctx=64), 77, "q4_k")
tokens = rng.integers(0, 768, 45).tolist()
ok, e = close(m.forward(tokens, 0), o.forward(tokens, 0))
assert ok, e
print("h6 ok")
"""


@pytest.mark.parametrize("shape,splits", [("8,7", 1), ("8,6", 1), ("4,4", 1), ("8,7", 2), ("4,4", 4)])
def test_gemm_on_f16_and_fp6_operands(shape, splits):
    env = dict(os.environ, JQ_GEMM_H6_SHAPE=shape, JQ_GEMM_H6_SPLITS=str(splits), JQ_GEMM_H6_MIN_M="17", JQ_Q4K_NO_ROWS16="1")
    res = subprocess.run([sys.executable, "-c", CHILD.replace("%r", repr(ROOT), 1)], env=env, capture_output=True, text=True, timeout=110)
    assert res.returncode == 0 and "h6 ok" in res.stdout, res.stdout + res.stderr


@pytest.mark.parametrize("splits", [1, 4])
def test_workgroups_of_eight_groups_of_weight_rows(splits):
    test_gemm_on_f16_and_fp6_operands("8,8", splits)


def q4k_blocks(d, dmin, sc, mn, q):
    """Blocks of [n][super-blocks]: d, dmin, sc and mn [..., 8] of six bits, q [..., 8, 32] of four."""
    b = np.zeros(d.shape + (144,), np.uint8)
    b[..., 0:2] = d.astype(np.float16)[..., None].view(np.uint8)
    b[..., 2:4] = dmin.astype(np.float16)[..., None].view(np.uint8)
    b[..., 4:8] = sc[..., :4] | sc[..., 4:] >> 4 << 6
    b[..., 8:12] = mn[..., :4] | mn[..., 4:] >> 4 << 6
    b[..., 12:16] = (sc[..., 4:] & 15) | (mn[..., 4:] & 15) << 4
    b[..., 16:] = (q[..., 0::2, :] | q[..., 1::2, :] << 4).reshape(d.shape + (128,))
    return b.reshape(-1)


@pytest.mark.parametrize("scales", ["at most 1", "at most 2", "at most 4", "at most 8", "at most 63", "all 1", "all 31", "all 63", "one of 1"])
def test_error_whatever_the_weights_scales(scales):
    """Super-blocks whose six-bit scales are small, and activations that meet a small scale among large ones: the error against 64
    bits does not depend on them.  The weights lie about zero (dmin m = 8 d sc), so that the codes' product is all of the result.

    In root mean square the remainder l is at most 2^-10 / sqrt(12) of its activation (f16), and E2M3 takes at most 2^-3 / sqrt(12) of
    each of its product's two factors: sqrt(2) / 12 2^-13 = 1.44e-5 of the result.  (Factors below E2M3's normal numbers lose
    more of themselves, and are that much less of the sum.)"""
    rng = np.random.default_rng(17)
    m, k, n = 160, 2048, 1024
    t = 63 if scales == "one of 1" else int(scales.split()[-1])
    sc = np.full((n, k // 256, 8), t, np.uint8) if scales.startswith("all") else rng.integers(1, t + 1, (n, k // 256, 8), dtype=np.uint8)
    x = rng.standard_normal((m, k)).astype(np.float32)
    if scales == "one of 1":
        sc[:, :, 3] = 1
        x.reshape(m, -1, 8, 32)[:, :, [0, 1, 2, 4, 5, 6, 7]] *= np.float32(2e-5)
    d = rng.uniform(1e-4, 1e-3, (n, k // 256)).astype(np.float16)
    mn = np.round(sc * (63.0 / t)).astype(np.uint8)
    q = rng.integers(0, 16, (n, k // 256, 8, 32), dtype=np.uint8)
    blocks = q4k_blocks(d, d.astype(np.float64) * 8 * t / 63, sc, mn, q)
    got = capi.Weight.upload(capi.Q4_K, blocks, n, k).matmul_t(m, x)
    want = x.astype(np.float64) @ oracle.dequantize(capi.Q4_K, blocks).reshape(n, k).astype(np.float64).T
    rel = np.sqrt(((got - want) ** 2).mean() / (want ** 2).mean())
    assert rel <= 1.45e-5, float(rel)


@pytest.mark.parametrize("qtype,m,k,n,kernel,arithmetic", [
    (capi.Q4_K, 127, 4096, 14336, "q4k_gemm_i8", "int8"), (capi.Q4_K, 128, 4096, 14336, "q4k_gemm_i8", "f16+fp6"),
    (capi.Q4_K, 512, 4096, 14336, "q4k_gemm_i8", "f16+fp6"), (capi.Q4_K, 128, 4096, 256, "q4k_gemm_mfma", ""),
    (capi.Q6_K, 512, 4096, 1024, "q6k_gemm_i8", "int8"), (capi.Q4_K, 1, 4096, 4096, "q4k_gemv_mfma_lds", "")])
def test_arithmetic_chosen_for_a_shape(qtype, m, k, n, kernel, arithmetic):
    import torch
    w = capi.Weight.upload(qtype, np.zeros(n * k // 256 * (144 if qtype == capi.Q4_K else 210), np.uint8), n, k)
    x, y = torch.zeros(m * k, device="cuda"), torch.empty(m * n, device="cuda")
    w.matmul_t_dev(m, x.data_ptr(), m * k, y.data_ptr(), m * n, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    assert (capi.last_kernel().split("+")[0], capi.last_arithmetic()) == (kernel, arithmetic)


def device_product(call, m, k, n, x, stream):
    import torch
    y = torch.full((m, n), float("nan"), device="cuda")
    call(m, x.data_ptr(), m * k, y.data_ptr(), m * n, stream)
    return y


@pytest.mark.parametrize("m,k,n,whole", [(128, 4096, 1024, True), (300, 2048, 2000, True), (900, 4096, 4096, True), (3072, 4096, 4096, True),
                                         (1024, 12288, 4096, False), (1077, 12288, 640, False), (130, 98304, 256, False)])
def test_the_call_that_allocates_nothing_takes_the_same_arithmetic(m, k, n, whole):
    """Also where the prepared activations of all rows do not fit its scratch (from m k = 11.1M elements on; above 14.8M it fails).
    `whole`: both calls split k alike, so that not even the order of a sum differs."""
    import torch
    blocks = synth.normal_quantized(capi.Q4_K, 61, n * k, 0.02)
    w = capi.Weight.upload(capi.Q4_K, blocks, n, k)
    x = torch.from_numpy(synth.normal(62, (m, k))).cuda()
    s = torch.cuda.current_stream().cuda_stream
    ref = device_product(w.matmul_t_dev, m, k, n, x, s)
    names = [(capi.last_kernel(), capi.last_arithmetic())]
    new = device_product(w.matmul_t_noalloc, m, k, n, x, s)
    names.append((capi.last_kernel(), capi.last_arithmetic()))
    torch.cuda.synchronize()
    assert [a for _, a in names] == ["f16+fp6"] * 2, names
    if whole:
        assert torch.equal(ref, new), names
    wd = torch.from_numpy(oracle.dequantize(capi.Q4_K, blocks).reshape(n, k)).cuda().double()
    want = x.double() @ wd.T
    for got in (ref, new):
        assert ((got - want).square().mean() / want.square().mean()).sqrt().item() <= 1.45e-5


def test_capture_on_a_stream_that_never_ran_a_product_of_that_size():
    """Scratch between 64 and 128 MB (114 here): a cold stream can be captured, as it can above."""
    import torch
    m, k, n = 3072, 12288, 256
    w = capi.Weight.upload(capi.Q4_K, synth.normal_quantized(capi.Q4_K, 63, n * k, 0.02), n, k)
    x = torch.from_numpy(synth.normal(64, (m, k))).cuda()
    want = device_product(w.matmul_t_dev, m, k, n, x, torch.cuda.current_stream().cuda_stream)
    torch.cuda.synchronize()
    stream, y = torch.cuda.Stream(), torch.full((m, n), float("nan"), device="cuda")
    graph = torch.cuda.CUDAGraph()
    torch.cuda.synchronize()
    with torch.cuda.graph(graph, stream=stream):
        w.matmul_t_dev(m, x.data_ptr(), m * k, y.data_ptr(), m * n, stream.cuda_stream)
    for _ in range(3):
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y, want)
        device_product(w.matmul_t_dev, m, k, n, x, torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
    del graph
    torch.cuda.synchronize()
    capi.stream_release(stream.cuda_stream)


MX_CHILD = r"""
import os, sys
import numpy as np
sys.path.insert(0, ROOT)
import oracle
from joshua_amd import capi, synth
splits = int(os.environ["JQ_GEMM_H6_SPLITS"])


def check(blocks, lhs, what, rms=None):
    # the weights are exact, E2M1 in both instructions; a remainder, at most 8 s for s = 2^-14 of its super-block's largest magnitude, is
    # at most s / 2 off as E2M3; f32 sums: 2^-20 of the terms
    m, k = lhs.shape
    n = blocks.size // (k // 32 * 17)
    got = capi.Weight.upload(capi.MXFP4, blocks, n, k).matmul_t(m, lhs)
    assert capi.last_kernel() == "mxfp4_gemm_i8" + ("+splitk" if splits > 1 else "") and capi.last_arithmetic() == "f16+fp6"
    w, x = oracle.dequantize(capi.MXFP4, blocks).reshape(n, k).astype(np.float64), lhs.astype(np.float64)
    want = x @ w.T
    s = np.abs(x.reshape(m, -1, 256)).max(2) * 2.0 ** -14
    bound = 0.5 * s @ np.abs(w).reshape(n, -1, 256).sum(2).T + 2.0 ** -20 * (np.abs(x) @ np.abs(w).T)
    err = np.abs(got - want)
    assert np.all(err <= bound), (what, float((err / np.maximum(bound, 1e-300)).max()))
    if rms:
        assert np.sqrt((err ** 2).mean() / (want ** 2).mean()) <= rms, what
    return got


sizes = [(17, 256, 64), (33, 512, 113), (64, 1024, 97), (129, 768, 112), (257, 512, 300), (256, 1024, 96)] if splits == 1 else [(40, 4096, 100), (300, 4096, 130)]
for m, k, n in sizes:
    check(synth.normal_quantized(capi.MXFP4, 5 + n, n * k, 0.02), synth.normal(6 + k, (m, k)), (m, k, n), 1.2e-5)
rng = np.random.default_rng(4)
n, k = 80, 2304 if splits == 1 else 4096
raw = rng.integers(0, 256, (n * k // 32, 17), dtype=np.uint8)
raw[:, 0] = rng.integers(105, 145, len(raw))
raw[::13, 0], raw[::17, 0], raw[:8, 0] = 0xFF, 0, 0xFF
lhs = synth.normal(9, (50, k))
lhs[0] *= (10.0 ** rng.integers(-6, 7, size=k // 16)).repeat(16).astype(np.float32)
lhs[1] = 0
lhs[1, 1234] = 3.5
lhs[3] *= np.float32(1e25)
got = check(raw.reshape(-1), lhs, "every scale")
lhs[7, 100], lhs[8, 2000] = np.inf, np.nan
other = capi.Weight.upload(capi.MXFP4, raw.reshape(-1), n, k).matmul_t(50, lhs)
assert np.all(np.isnan(other[7:9])) and np.array_equal(np.delete(other, [7, 8], 0), np.delete(got, [7, 8], 0))
print("h6 ok")
"""


@pytest.mark.parametrize("shape,splits", [("8,8", 1), ("8,7", 1), ("8,6", 1), ("4,4", 1), ("8,8", 4), ("4,4", 2)])
def test_mxfp4_on_f16_and_its_own_codes(shape, splits):
    env = dict(os.environ, JQ_GEMM_H6_SHAPE=shape, JQ_GEMM_H6_SPLITS=str(splits), JQ_GEMM_H6_MIN_M="17")
    res = subprocess.run([sys.executable, "-c", MX_CHILD.replace("ROOT", repr(ROOT), 1)], env=env, capture_output=True, text=True, timeout=110)
    assert res.returncode == 0 and "h6 ok" in res.stdout, res.stdout + res.stderr


@pytest.mark.parametrize("m,k,n", [(200, 4096, 4096), (333, 2304, 2112)])
def test_mxfp4_activations_that_few_bits_hold(m, k, n):
    """Magnitudes that are all alike, one element in 256, the largest's halves and quarters, bf16 values: held whole, so the products lie f32
    roundings off; normal ones as far as f16 and an E2M3 remainder are (8 s for s = 2^-14 of the largest, s / 2 off)."""
    blocks, rng = synth.normal_quantized(capi.MXFP4, 80, n * k, 0.02), np.random.default_rng(81)
    w, d = capi.Weight.upload(capi.MXFP4, blocks, n, k), oracle.dequantize(capi.MXFP4, blocks).reshape(n, k).astype(np.float64)
    normal = rng.standard_normal((m, k)).astype(np.float32)
    one = np.zeros((m, k), np.float32)
    one[:, 77::256] = normal[:, 77::256]
    size = rng.uniform(0.5, 2, (m, 1)).astype(np.float32)
    for what, x, bound in (("alike", np.sign(normal) * size, 2e-7), ("one", one, 2e-7),
                           ("halves", np.sign(normal) * size * rng.choice([1.0, 0.5, 0.25], (m, k)).astype(np.float32), 2e-7),
                           ("bf16", (normal.view(np.uint32) & 0xFFFF0000).view(np.float32), 2e-7), ("normal", normal, 7e-6)):
        got = w.matmul_t(m, np.ascontiguousarray(x, dtype=np.float32))
        assert capi.last_arithmetic() == "f16+fp6"
        want = x.astype(np.float64) @ d.T
        err = np.linalg.norm(got - want) / np.linalg.norm(want)
        assert err <= bound, (what, err)
