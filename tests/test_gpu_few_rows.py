"""Products of up to some 100 activation rows on pairs of f16 numbers (few_rows, few_rows_many) against 64-bit products of the decoded weights."""
import os
import subprocess
import sys

import numpy as np
import pytest

import oracle
from joshua_amd import capi, synth

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
ON = not os.environ.get("JQ_FEW_ROWS", "1").startswith("0")
TYPES = [capi.Q4_K, capi.Q6_K, capi.Q8_0, capi.MXFP4]


def check(qtype, blocks, n, k, lhs, rms=3e-7, w=None):
    """An activation s (hi + lo) is at most 2^-22 of itself off (2^-38 of its super-block's largest), the product of the two remainders,
    left out, 2^-22 of the whole; f32 sums: some 8 roundings a super-block, a dozen of those, 8 waves, within a matrix instruction up to
    four a result: 2^-18 of the terms' magnitudes in all.  Q4_K's terms are those of sc (q - 8) and of what it leaves."""
    m = len(lhs)
    got = (w or capi.Weight.upload(qtype, blocks, n, k)).matmul_t(m, lhs)
    assert capi.last_arithmetic() == "f16 pairs", (capi.last_kernel(), capi.last_arithmetic())
    d, x = oracle.dequantize(qtype, blocks).reshape(n, k).astype(np.float64), lhs.astype(np.float64)
    mag = np.abs(d)
    if qtype == capi.Q4_K:
        b = blocks.reshape(n, k // 256, 144)
        s = b[:, :, 4:16].astype(np.int64)
        sc = np.concatenate([s[:, :, :4] & 63, (s[:, :, 8:] & 15) | s[:, :, :4] >> 6 << 4], 2)
        mn = np.concatenate([s[:, :, 4:8] & 63, s[:, :, 8:] >> 4 | s[:, :, 4:8] >> 6 << 4], 2)
        f = np.abs(b[:, :, 0:4].copy().view(np.float16).astype(np.float64))
        mag = mag + 2 * (8 * f[:, :, :1] * sc + f[:, :, 1:] * mn).repeat(32, 2).reshape(n, k)
    top = np.abs(x.reshape(m, -1, 256)).max(2).repeat(256, 1)
    want, err = x @ d.T, None
    err = np.abs(got - want)
    bound = 2.0 ** -18 * (np.abs(x) @ mag.T) + 2.0 ** -36 * (top @ mag.T)
    assert np.all(err <= bound), (m, k, n, float((err / np.maximum(bound, 1e-300)).max()))
    if rms:
        assert np.sqrt((err ** 2).mean() / (want ** 2).mean()) <= rms
    return got


# a tile of 16 weight rows a workgroup, two, four; their ragged ends; rows of 8 to 17 super-blocks over up to 8 waves
@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("m,k,n", [(3, 2304, 2049), (4, 2048, 1295), (5, 4352, 1024), (8, 2560, 4097), (9, 2048, 5001), (16, 2304, 8223),
                                   (16, 2048, 12289), (7, 1280, 12337), (13, 1280, 16399)])
def test_edges_of_tiles(qtype, m, k, n):
    blocks = synth.normal_quantized(qtype, 5 + n, n * k, 0.02)
    check(qtype, blocks, n, k, synth.normal(6 + k, (m, k)))


MANY = r"""
import sys
sys.path.insert(0, %r)
from joshua_amd import capi, synth
from tests.test_gpu_few_rows import TYPES, check
for m, k, n in [(17, 2304, 1025), (33, 2048, 1039), (48, 4352, 1024), (64, 1280, 2111), (65, 2048, 1100), (127, 2304, 1055)]:
    for qtype in TYPES:
        check(qtype, synth.normal_quantized(qtype, 5 + n, n * k, 0.02), n, k, synth.normal(6 + k, (m, k)))
print("many ok")
"""


@pytest.mark.parametrize("shape", ["1,2", "2,2", "4,2", "2,3", "2,4"])
def test_more_than_16_rows_in_every_workgroup_shape(shape):
    """The shape is read at the first product, hence the child process."""
    res = subprocess.run([sys.executable, "-c", MANY % ROOT], env=dict(os.environ, JQ_FEW_ROWS_SHAPE=shape), capture_output=True, text=True, timeout=110)
    assert res.returncode == 0 and "many ok" in res.stdout, res.stdout + res.stderr


@pytest.mark.parametrize("qtype,m,k,n", [(capi.Q4_K, 61, 7168, 2112), (capi.Q6_K, 100, 4096, 4096), (capi.Q8_0, 40, 2304, 1500), (capi.MXFP4, 160, 2048, 1024)])
def test_the_call_that_allocates_nothing(qtype, m, k, n):
    import torch
    w = capi.Weight.upload(qtype, synth.normal_quantized(qtype, 61, n * k, 0.02), n, k)
    x, y = torch.from_numpy(synth.normal(62, (m, k))).cuda(), torch.full((2, m, n), float("nan"), device="cuda")
    s = torch.cuda.current_stream().cuda_stream
    for i, call in enumerate((w.matmul_t_dev, w.matmul_t_noalloc)):
        call(m, x.data_ptr(), m * k, y[i].data_ptr(), m * n, s)
        assert (capi.last_kernel(), capi.last_arithmetic()) == ("few_rows_many", "f16 pairs")
    torch.cuda.synchronize()
    assert torch.equal(y[0], y[1])


@pytest.mark.parametrize("qtype,k,n", [(capi.Q8_0, 5120, 2561), (capi.MXFP4, 4096, 4096), (capi.Q6_K, 7936, 8460)])
def test_one_row_that_no_other_kernel_takes(qtype, k, n):
    check(qtype, synth.normal_quantized(qtype, 7, n * k, 0.02), n, k, synth.normal(8, (1, k)))


@pytest.mark.parametrize("qtype,step", [(capi.Q6_K, 210), (capi.MXFP4, 136)])
def test_blocks_at_every_offset_to_16_bytes(qtype, step):
    """Rows of an odd number of super-blocks from an offset into the allocation, up to its last byte."""
    k, n = 9 * 256, 1100
    raw = synth.normal_quantized(qtype, 9, (n * 9 + 3) * 256, 0.02)
    parent = capi.Weight.upload(qtype, raw, n * 9 + 3, 256)
    lhs = synth.normal(10, (6, k))
    for first in (1, 2, 3):
        for rows in (lhs, np.concatenate([lhs] * 4)):
            check(qtype, raw[first * step:first * step + n * 9 * step], n, k, rows, w=parent.view(first * step, n, k))


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("m", [5, 12, 40])
def test_every_scale_and_rows_of_every_range(qtype, m):
    n, k = 1040, 2304
    rng = np.random.default_rng(3)
    if qtype == capi.Q8_0:
        raw = rng.integers(0, 256, (n * k // 32, 34), dtype=np.uint8)
        raw[:, :2] = (rng.uniform(-1, 1, len(raw)) * 2.0 ** rng.integers(-12, 1, len(raw))).astype(np.float16)[:, None].view(np.uint8)
        raw[::11, :2] = 0
        raw[:8, :2] = 0
    elif qtype == capi.MXFP4:
        raw = rng.integers(0, 256, (n * k // 32, 17), dtype=np.uint8)
        raw[:, 0] = rng.integers(110, 140, len(raw))
        raw[::13, 0] = 0xFF   # stands for zeros
        raw[::17, 0] = 0
        raw[:8, 0] = 0xFF
    else:
        size, at = (144, [0, 2]) if qtype == capi.Q4_K else (210, [208])
        raw = rng.integers(0, 256, (n * k // 256, size), dtype=np.uint8)
        for i in at:
            raw[:, i:i + 2] = (rng.uniform(-1, 1, len(raw)) * 1e-3).astype(np.float16)[:, None].view(np.uint8)
        raw[::7, at[0]:at[0] + 2] = 0
    lhs = synth.normal(9, (m, k))
    lhs[0] *= (10.0 ** rng.integers(-6, 7, size=k // 16)).repeat(16).astype(np.float32)
    lhs[1] = 0
    lhs[1, 1234] = 3.5
    lhs[2, 512:1024] = 0
    lhs[3] *= np.float32(1e30)
    lhs[4] *= np.float32(1e-30)
    got = check(qtype, raw.reshape(-1), n, k, lhs, rms=None)
    lhs[0, 100], lhs[2, 2000] = np.inf, np.nan
    other = capi.Weight.upload(qtype, raw.reshape(-1), n, k).matmul_t(m, lhs)
    assert not np.isfinite(other[[0, 2]]).any()
    assert np.array_equal(np.delete(other, [0, 2], 0), np.delete(got, [0, 2], 0))


@pytest.mark.parametrize("qtype", TYPES)
@pytest.mark.parametrize("m", [5, 12, 40])
def test_rows_up_to_the_ends_of_f32(qtype, m):
    """Activations behind no power of two within 2^100 of 1: each row as exact as one of ordinary size."""
    n, k = 1040, 2304
    blocks = synth.normal_quantized(qtype, 5, n * k, 0.01)
    lhs = synth.normal(6, (m, k))
    lhs /= np.abs(lhs).max(1, keepdims=True)
    for i, size in enumerate((1.0, 1e35, 3e38, 1e-36)):
        lhs[i] *= np.float32(size)
    got = check(qtype, blocks, n, k, lhs, rms=None).astype(np.float64)
    want = lhs.astype(np.float64) @ oracle.dequantize(qtype, blocks).reshape(n, k).astype(np.float64).T
    assert np.all(np.linalg.norm(got - want, axis=1) <= 3e-7 * np.linalg.norm(want, axis=1))


@pytest.mark.parametrize("qtype", [capi.Q8_0, capi.MXFP4])
@pytest.mark.parametrize("m,k,n", [(5, 2304, 1040), (12, 2304, 1040), (16, 2048, 12289), (40, 2304, 1040), (127, 2304, 1055)])
def test_blocks_whose_scales_lie_far_below_their_neighbours(qtype, m, k, n):
    """Block j of every super-block behind the j-th of eight scales up to 2^190 (MXFP4) or 2^38 apart, activation row i zero but for one block
    each: as exact as if that were alone, on either side of what one f16 operand holds (2^26 and 2^21)."""
    if qtype == capi.MXFP4:
        raw = np.array(synth.normal_quantized(qtype, 5, n * k, 0.02)).view(np.uint8).reshape(n, k // 256, 8, 17)
        raw[..., 0] = [200, 173, 174, 127, 90, 40, 199, 10]
    else:
        raw = np.array(synth.normal_quantized(qtype, 5, n * k, 0.02)).view(np.uint8).reshape(n, k // 256, 8, 34)
        d = np.random.default_rng(6).uniform(1, 2, (n, k // 256, 8)) * 2.0 ** np.array([14, -7, -8, -14, -18, 0, 13, -23])
        raw[..., :2] = d.astype(np.float16)[..., None].view(np.uint8)
    lhs = synth.normal(7, (m, k)).reshape(m, k // 256, 8, 32)
    lhs = np.where(np.arange(8)[:, None] == np.arange(m)[:, None, None, None] % 8, lhs, np.float32(0)).reshape(m, k)
    blocks = raw.reshape(-1)
    got = capi.Weight.upload(qtype, blocks, n, k).matmul_t(m, lhs).astype(np.float64)
    assert capi.last_arithmetic() == "f16 pairs"
    want = lhs.astype(np.float64) @ oracle.dequantize(qtype, blocks).reshape(n, k).astype(np.float64).T
    assert np.all(np.linalg.norm(got - want, axis=1) <= 3e-7 * np.linalg.norm(want, axis=1))


@pytest.mark.parametrize("m", [5, 12, 40])
@pytest.mark.parametrize("scale,size", [(240, 1e-30), (250, 1e-36), (5, 1e35)])
def test_mxfp4_scales_at_the_ends_of_their_range(m, scale, size):
    n, k = 1040, 2304
    raw = np.array(synth.normal_quantized(capi.MXFP4, 5, n * k, 0.02)).view(np.uint8).reshape(-1, 17)
    raw[:, 0] = scale
    lhs = synth.normal(6, (m, k)) * np.float32(size)
    got = capi.Weight.upload(capi.MXFP4, raw.reshape(-1), n, k).matmul_t(m, lhs).astype(np.float64)
    assert capi.last_arithmetic() == "f16 pairs"
    want = lhs.astype(np.float64) @ oracle.dequantize(capi.MXFP4, raw.reshape(-1)).reshape(n, k).astype(np.float64).T
    assert np.linalg.norm(got - want) <= 3e-7 * np.linalg.norm(want)


@pytest.mark.parametrize("qtype,bound", [(capi.Q8_0, 1.22e-7), (capi.Q6_K, 1.53e-7), (capi.MXFP4, 1.20e-7)])
@pytest.mark.parametrize("m", [2, 5, 12])
def test_no_further_off_than_the_f32_row_kernels(qtype, bound, m):
    """Rows of 2048, where those have the fewest roundings; the bound is what they lie off on the same inputs."""
    n, k = 3072, 2048
    err = ref = 0.0
    for seed in range(4):
        blocks, lhs = synth.normal_quantized(qtype, 90 + seed, n * k, 0.02), synth.normal(95 + seed, (m, k))
        got = capi.Weight.upload(qtype, blocks, n, k).matmul_t(m, lhs)
        assert capi.last_arithmetic() == ("f16 pairs" if ON else "")
        want = lhs.astype(np.float64) @ oracle.dequantize(qtype, blocks).reshape(n, k).astype(np.float64).T
        err, ref = err + ((got - want) ** 2).sum(), ref + (want ** 2).sum()
    assert np.sqrt(err / ref) <= bound, np.sqrt(err / ref)


@pytest.mark.parametrize("qtype,m,k,n,kernel", [
    (capi.Q6_K, 2, 4096, 1024, "matmul_rows_staged"), (capi.Q6_K, 3, 4096, 1536, "matmul_rows_staged"), (capi.Q6_K, 5, 12288, 1024, "matmul_rows_staged"),
    (capi.Q8_0, 1, 9984, 1024, "matmul_rows_staged"), (capi.Q8_0, 2, 4096, 1024, "matmul_rows_staged"), (capi.Q8_0, 2, 12288, 2048, "q8_0_gemv_dot4_lds"),
    (capi.Q6_K, 2, 12288, 2048, "q6k_gemv_mfma_cols"), (capi.MXFP4, 1, 16384, 1024, "matmul_rows_staged"),
    (capi.Q6_K, 2, 4096, 3072, None), (capi.Q6_K, 6, 4096, 1024, None), (capi.Q8_0, 2, 4096, 1280, None), (capi.MXFP4, 2, 4096, 1024, None)])
def test_few_weight_rows_keep_the_kernels_that_are_faster_there(qtype, m, k, n, kernel):
    blocks, lhs = synth.normal_quantized(qtype, 70, n * k, 0.02), synth.normal(71, (m, k))
    got = capi.Weight.upload(qtype, blocks, n, k).matmul_t(m, lhs)
    assert capi.last_kernel() == kernel if kernel else capi.last_arithmetic() == "f16 pairs"
    want = oracle.matmul_t(qtype, (m, k, n), lhs, blocks, avx2=oracle.have_avx2())
    assert np.all(np.abs(got - want) <= 1e-3 * np.maximum(np.abs(want), 1.0))


@pytest.mark.parametrize("qtype,m,k,n,kernel", [
    (capi.Q4_K, 127, 1024, 14336, "q4k_gemm_i8"), (capi.Q6_K, 128, 2304, 14336, "q6k_gemm_i8"), (capi.Q8_0, 127, 1024, 14336, "q8_0_gemm_i8"),
    (capi.MXFP4, 128, 2304, 14336, "mxfp4_gemm_i8"), (capi.MXFP4, 160, 1024, 24576, "mxfp4_gemm_i8"), (capi.Q6_K, 200, 7168, 576, "q6k_gemm_i8+splitk"),
    (capi.Q4_K, 64, 1024, 9000, "few_rows_many"), (capi.Q6_K, 144, 9984, 700, "few_rows_many"), (capi.Q8_0, 80, 2048, 11008, "few_rows_many"),
    (capi.MXFP4, 130, 9984, 1500, "few_rows_many")])
def test_some_hundred_rows_go_where_they_are_faster(qtype, m, k, n, kernel):
    """Shapes on either side of the line between few_rows_many and the GEMMs behind it, each at least a sixth slower on the other."""
    blocks, lhs = synth.normal_quantized(qtype, 72, n * k, 0.02), synth.normal(73, (m, k))
    got = capi.Weight.upload(qtype, blocks, n, k).matmul_t(m, lhs)
    assert capi.last_kernel() == kernel or not ON
    want = lhs.astype(np.float64) @ oracle.dequantize(qtype, blocks).reshape(n, k).astype(np.float64).T
    assert np.all(np.abs(got - want) <= 1e-3 * np.maximum(np.abs(want), 1.0))
