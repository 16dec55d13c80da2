"""Products with plain bf16 rows in tiles of 256 activation rows (one workgroup a compute unit): one run of k and several, row and column counts
at the edges of the tiles and within them, alone and in a gated feed-forward block."""
import os
import subprocess
import sys

import numpy as np
import pytest

from joshua_amd import capi
from joshua_amd.synth import layered as sl
from joshua_amd.synth import normal
from tests import layered_cases as lc
from tests.layered_cases import build, check, feed, tokens

pytestmark = pytest.mark.gpu

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("m,n,k,kernel", [
    (512, 4096, 4096, "dense_gemm_wide+splitk"),
    (449, 6141, 4090, "dense_gemm_wide+splitk"),     # the last row tile of 193 rows; columns and k within a tile and a stage
    (257, 24575, 2048, "dense_gemm_wide"),           # one row more than a tile
    (1985, 7681, 2090, "dense_gemm_wide"),           # a column tile of one column
    (512, 16000, 4096, "dense_gemm"),                # two full rounds of the smaller tiles
])
def test_products_of_many_rows(m, n, k, kernel):
    """Against 64 bits on the operands as the matrix cores take them; f32 sums of k exact products, 2^-24 of the terms' magnitudes
    for each of some tens of roundings of a sum's size."""
    w, x = sl.to_bf16(normal(1, (n, k), k ** -0.5)), normal(2, (m, k))
    got = capi.Weight.upload(capi.BF16, w, n, k).matmul_t(m, x)
    assert capi.last_kernel() == kernel
    rows = sorted({r for r in (0, 1, 17, 100, 127, 128, 192, 254, 255, 256, 257, 300, m - 2, m - 1) if r < m})
    x, w = sl.from_bf16(sl.to_bf16(x[rows])).astype(np.float64), sl.from_bf16(w).astype(np.float64)
    scale = np.abs(x) @ np.abs(w).T
    assert np.all(np.abs(got[rows] - x @ w.T) <= 2e-6 * scale + 1e-7)


@pytest.mark.parametrize("m,n,k,kernel", [
    (64, 24571, 2048, "dense_gemm+splitk"),    # 192 tiles of 128 weight rows, the last of them ragged: two runs
    (61, 24571, 2530, "dense_gemm+splitk"),    # four runs of 10 stages, the last one part-filled
    (9, 32640, 1090, "dense_gemm+splitk"),     # 255 tiles: two runs of 9 stages
    (17, 32640, 4000, "dense_gemm+splitk"),    # 63 stages, of which two runs would begin 4096 bytes apart: three
    (64, 32640, 1984, "dense_gemm"),           # 31 stages: the sums of 64 rows would cost more
    (33, 32769, 1024, "dense_gemm"),           # 257
    (65, 24571, 1024, "dense_gemm"),           # a second tile of rows
    (20, 24571, 900, "dense_gemm"),            # 15 stages
])
def test_products_of_one_tile_of_rows(m, n, k, kernel):
    """As above, of up to 64 rows, which wait for the weights."""
    w, x = sl.to_bf16(normal(3, (n, k), k ** -0.5)), normal(4, (m, k))
    got = capi.Weight.upload(capi.BF16, w, n, k).matmul_t(m, x)
    assert capi.last_kernel() == kernel
    x, w = sl.from_bf16(sl.to_bf16(x)).astype(np.float64), sl.from_bf16(w).astype(np.float64)
    scale = np.abs(x) @ np.abs(w).T
    assert np.all(np.abs(got - x @ w.T) <= 2e-6 * scale + 1e-7)


@pytest.mark.parametrize("rows", [9, 64])
def test_gated_block_of_one_tile_of_rows(tmp_path, rows):
    cfg = lc.model(2048, 40, [lc.dense(lc.mamba(16, 2, 2, 2), 12283, limit=0.4)])
    m, o, _ = build(tmp_path, cfg, 23, lc.BF16, n_ctx=512)
    toks = tokens(cfg, 24, rows)
    check(feed(m, toks, []), o.forward(toks), lc.BF16, "whole", o)


def test_one_tile_of_rows_is_not_split_in_two():
    w = capi.Weight.upload(capi.BF16, np.zeros(24576 * 4096, np.uint16), 24576, 4096)
    for m, kernel in ((200, "dense_gemm"), (300, "dense_gemm_wide")):
        w.matmul_t(m, np.ones((m, 4096), np.float32))
        assert capi.last_kernel() == kernel


@pytest.mark.parametrize("ff", [12283, 4096])
def test_gated_block_of_many_rows(tmp_path, ff):
    """A feed-forward block whose gate and up rows run in one launch, whole and in runs of k."""
    cfg = lc.model(2048 if ff > 10000 else 4096, 40, [lc.dense(lc.mamba(16, 2, 2, 2), ff, limit=0.4)])
    m, o, _ = build(tmp_path, cfg, 21, lc.BF16, n_ctx=512)
    toks = tokens(cfg, 22, 500)
    check(feed(m, toks, []), o.forward(toks), lc.BF16, "whole", o)


CHILD = r"""
import sys
sys.path.insert(0, ROOT)
import pathlib
import tempfile
import numpy as np
from joshua_amd import capi
from tests import layered_cases as lc
for ff, n_tokens in ((1283, 500), (1440, 270)):   # columns within a tile of 96 and of 128 gate rows, and where one ends; rows of the last tile
    cfg = lc.model(2048, 40, [lc.dense(lc.mamba(16, 2, 2, 2), ff, limit=0.4)])
    with tempfile.TemporaryDirectory() as folder:
        m, o, _ = lc.build(pathlib.Path(folder), cfg, 31, lc.BF16, n_ctx=512)
    toks = lc.tokens(cfg, 32, n_tokens)
    lc.check(lc.feed(m, toks, []), o.forward(toks), lc.BF16, ff, o)
w, x = np.full(4096 * 2048, 0x3F80, np.uint16), np.ones((300, 2048), np.float32)   # ones: every sum is 2048
got = capi.Weight.upload(capi.BF16, w, 4096, 2048).matmul_t(300, x)
assert capi.last_kernel() == "dense_gemm_wide" + ("+splitk" if RUNS > 1 else "") and np.all(got == 2048.0)
print("wide ok")
"""


@pytest.mark.parametrize("rows", [192, 256])
@pytest.mark.parametrize("runs", [1, 3])
def test_gated_block_in_every_tile_and_in_runs(rows, runs):
    """The shape is read at the first product, hence the child process; the feed-forward blocks have more than the 128 tiles of 64 x 128 from which
    a product may take it."""
    res = subprocess.run([sys.executable, "-c", CHILD.replace("ROOT", repr(ROOT), 1).replace("RUNS", str(runs))], capture_output=True, text=True, timeout=110,
                         env=dict(os.environ, JQ_DENSE_WIDE=f"{rows},{runs}"))
    assert res.returncode == 0 and "wide ok" in res.stdout, res.stdout + res.stderr


def test_capture_of_one_tile_of_rows_behind_a_larger_call():
    """100 rows need no sums, 64 have two runs' worth: a stream that ran the larger call can be captured over the smaller one."""
    import torch
    n, k = 24571, 2048
    w = capi.Weight.upload(capi.BF16, sl.to_bf16(normal(5, (n, k), k ** -0.5)), n, k)
    x = torch.from_numpy(normal(6, (100, k))).cuda()
    want, y = torch.empty(64, n, device="cuda"), torch.empty(100, n, device="cuda")

    def product(m, out, stream):
        w.matmul_t_dev(m, x.data_ptr(), m * k, out.data_ptr(), m * n, stream)

    product(64, want, torch.cuda.current_stream().cuda_stream)
    assert capi.last_kernel() == "dense_gemm+splitk"
    torch.cuda.synchronize()
    stream = torch.cuda.Stream()
    product(100, y, stream.cuda_stream)
    assert capi.last_kernel() == "dense_gemm"
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        product(64, y, stream.cuda_stream)
    for _ in range(3):
        y.fill_(float("nan"))
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(y[:64], want)
        product(64, torch.empty_like(want), torch.cuda.current_stream().cuda_stream)
        torch.cuda.synchronize()
    del graph
    torch.cuda.synchronize()
    capi.stream_release(stream.cuda_stream)
