"""The block formats' matrix-core products at the edges of their tiles: 16
batch rows by 16 weight rows with K split over 4, 8 or 16 waves, and 32 or 64 batch
rows by 32, 64 or 128 weight rows with K split over 8, in 32-element sub-blocks.
Tests that are meant for one of them ask the launch rule that it takes their sizes.
Reference: the session's own dequantized weights (bit-identical
to the oracle's, test_gpu_formats.py) times x in f64. Bound: exact codes and
x to 2^-25, fp32 sums over K/32 sub-blocks of a wave: a few 2^-24, 2e-6 with the
cancellation of N(0, 1) inputs."""
import ctypes
import time

import numpy as np
import pytest

import launch_rules
from format_blocks import random_blocks
from test_gpu_dense import rel_l2

pytestmark = pytest.mark.gpu

FORMATS = [1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 16, 17]
SUPER = {6, 7, 8, 9, 10, 17}


def weights(rng, out, inp):
    """Rows of different magnitudes, not centred on zero."""
    W = rng.standard_normal((out, inp)) / np.sqrt(inp) + 0.3 / np.sqrt(inp)
    return (W * np.exp(rng.uniform(-3, 3, (out, 1)))).astype(np.float32)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("batch,inp,out", [
    (8, 256, 33),      # the least batch; one weight row past a tile
    (31, 768, 64),     # 24 sub-blocks over 8 waves
    (32, 1280, 16),    # as many weight rows as a tile
    (33, 512, 97),     # three 16-row blocks, ragged weight tile
    (97, 256, 200),    # last 16-row block nearly empty
    (385, 256, 1800),  # 64 x 64 tiles, ragged on both sides
    (200, 512, 6100),  # 64 x 128 tiles
])
def test_format_gemm_matches_f64(gpu, fmt, batch, inp, out):
    if fmt not in SUPER:
        inp += 96  # a number of sub-blocks that no wave count divides
    check_against_f64(gpu, fmt, batch, inp, out)


def check_against_f64(gpu, fmt, batch, inp, out):
    rng = np.random.default_rng(fmt * 1000 + batch + out)
    s = gpu.FormatDenseSession(batch, inp, out, gpu.LINEAR, fmt, W=weights(rng, out, inp))
    x = rng.standard_normal((batch, inp)).astype(np.float32)
    x *= np.exp(rng.uniform(-6, 6, (batch, 1))).astype(np.float32)
    y, _ = s.execute(x)
    W = s.export_f32().astype(np.float64)
    s.close()
    want = x.astype(np.float64) @ W.T
    # every batch row and every weight row by itself, against its own scale
    scale = np.abs(x).astype(np.float64) @ np.abs(W).T
    assert np.max(np.abs(y - want) / scale) <= 1e-6
    assert rel_l2(y, want) <= 2e-6


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("batch,inp,out,tile", [
    (33, 3072, 2081, (1, 1)),   # two 32-row blocks, the second with one row
    (40, 2560, 1376, (1, 1)),
    (128, 512, 4096, (1, 2)),   # exact tiles
    (97, 512, 5601, (1, 2)),    # one row past the last block on both sides
    (385, 512, 1800, (2, 2)),
    (200, 512, 6100, (2, 4)),
])
def test_each_gemm_tile_matches_f64(gpu, fmt, batch, inp, out, tile):
    for i in (inp, inp + 96):
        p = launch_rules.format_plan(fmt, out, i, batch)
        assert (p.kernel, p.tm, p.tn) == (launch_rules.GEMM,) + tile
    test_format_gemm_matches_f64(gpu, fmt, batch, inp, out)


@pytest.mark.parametrize("fmt,batch,inp,out,shape", [
    (2, 9, 64, 33, (4, 2)), (8, 16, 256, 33, (4, 2)),
    (2, 17, 352, 40, (4, 3)), (5, 8, 288, 40, (4, 3)),  # (11 and 9 sub-blocks: 3 and 2 a wave)
    (3, 9, 512, 20, (4, 4)), (9, 16, 512, 20, (4, 4)),
    (1, 8, 768, 33, (8, 3)), (6, 20, 768, 33, (8, 3)), (7, 8, 768, 33, (8, 3)),
    (4, 16, 1024, 17, (8, 4)), (10, 16, 1024, 4161, (8, 4)), (6, 16, 1024, 4161, (8, 4)),
    (8, 16, 1024, 513, (16, 2)), (6, 8, 1024, 513, (16, 2)), (7, 40, 1024, 100, (16, 2)),
    (2, 16, 1280, 33, (16, 3)), (10, 12, 1536, 33, (16, 3)), (3, 16, 4672, 20, (16, 4)),
    (17, 16, 2048, 50, (16, 4)), (6, 16, 4096, 50, (16, 4)),
])
def test_each_small_product_shape_matches_f64(gpu, fmt, batch, inp, out, shape):
    """Every built (waves, sub-blocks ahead) of the 16 x 16 blocks."""
    p = launch_rules.format_plan(fmt, out, inp, batch)
    assert (p.kernel, p.waves, p.depth) == (launch_rules.ROWS,) + shape
    check_against_f64(gpu, fmt, batch, inp, out)


@pytest.mark.parametrize("fmt", [1, 8])
@pytest.mark.parametrize("out,kernel", [(40, launch_rules.ROWS), (80, launch_rules.GEMM)])
def test_format_gemm_epilogue_and_row_runs(gpu, fmt, out, kernel):
    """Bias and activation, and rows that the scratch holds in several runs
    (the allocation-free execute has 64 MiB): the same bits as one run."""
    rng = np.random.default_rng(fmt)
    batch, inp = 1000, 16384
    plan = launch_rules.format_plan(fmt, out, inp, batch)
    assert plan.kernel == kernel
    assert kernel == launch_rules.ROWS or plan.run_rows < batch
    bias = rng.standard_normal(out)
    s = gpu.FormatDenseSession(batch, inp, out, gpu.SILU, fmt, W=weights(rng, out, inp), bias=bias)
    x = rng.standard_normal((batch, inp)).astype(np.float32)
    pre, post = s.execute(x)
    W = s.export_f32().astype(np.float64)
    z = (x.astype(np.float64) @ W.T + bias).astype(np.float32)
    assert rel_l2(pre, z) <= 2e-6
    assert rel_l2(post, pre / (1 + np.exp(-pre.astype(np.float64)))) <= 1e-6
    h = gpu.Hip()
    dx, dp, dq = h.upload(x), h.malloc(pre.nbytes), h.malloc(pre.nbytes)
    s.execute_noalloc(batch, dx, dp, dq)
    h.sync()
    assert np.array_equal(h.download(dp, pre.shape), pre)
    assert np.array_equal(h.download(dq, pre.shape), post)
    for p in (dx, dp, dq):
        h.free(p)
    s.close()


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("out,kernel", [(70, launch_rules.ROWS), (5600, launch_rules.GEMM)])
def test_format_gemm_non_finite_inputs(gpu, fmt, out, kernel):
    """A row of x with an infinity, a NaN or values near the f32 maximum (whose
    bf16 terms overflow) gives the dequantized product's result there and
    leaves the other rows alone."""
    rng = np.random.default_rng(fmt + 50)
    batch, inp = 40, 512
    assert launch_rules.format_plan(fmt, out, inp, batch).kernel == kernel
    s = gpu.FormatDenseSession(batch, inp, out, gpu.LINEAR, fmt, W=weights(rng, out, inp))
    x = rng.standard_normal((batch, inp)).astype(np.float32)
    clean, _ = s.execute(x)
    W = s.export_f32()
    x[3, 17], x[9, 300], x[35, 5], x[36, 40] = np.inf, np.nan, -np.inf, np.finfo(np.float32).max
    y, _ = s.execute(x)
    s.close()
    keep = [r for r in range(batch) if r not in (3, 9, 35, 36)]
    assert np.array_equal(y[keep], clean[keep])
    with np.errstate(invalid="ignore", over="ignore"):
        want = x.astype(np.float64) @ W.astype(np.float64).T
    assert np.isnan(y[9]).all()
    for r in (3, 35):
        assert np.array_equal(np.isnan(y[r]), np.isnan(want[r]))
        assert np.array_equal(np.isposinf(y[r]), np.isposinf(want[r]))
    with np.errstate(over="ignore"):
        top = want[36].astype(np.float32)  # some of these overflow
    fits = np.isfinite(top)
    assert rel_l2(y[36][fits] / 1e38, top[fits] / 1e38) <= 2e-6
    assert np.array_equal(y[36][~fits], top[~fits])


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("batch,inp,out", [
    (6, 768, 448),    # below 8 rows, few products: the per-row kernel
    (7, 8192, 40),    # long rows, few of them: likewise
    (16, 512, 130),   # 4 waves
    (16, 1024, 513),  # 8 waves; one weight row past a block
    (17, 1024, 512),  # one batch row in the second block
    (100, 768, 160),  # 7 batch blocks, the last with 4 rows
    (33, 2048, 400),  # 16 waves, 3 batch blocks
    (40, 2048, 1360),  # 85 x 3 blocks, the last count below 256
    (40, 2048, 1376),  # 86 x 3
])
def test_format_small_products_match_f64(gpu, fmt, batch, inp, out):
    test_format_gemm_matches_f64(gpu, fmt, batch, inp, out)


@pytest.mark.parametrize("fmt", FORMATS)
@pytest.mark.parametrize("batch,out,kernel", [(16, 70, launch_rules.ROWS), (40, 5600, launch_rules.GEMM)])
def test_format_gemm_small_inputs(gpu, fmt, batch, out, kernel):
    """Inputs down to f32's least normals keep fp32's digits, beside rows of
    ordinary size, and zeros stay zeros: bf16 terms of a value end at 2^-133.
    Bound: the products' 2e-6, and from 2^-120 on the rounding of outputs near the
    least normal (2^-149 of 2^-126 and less)."""
    rng = np.random.default_rng(fmt)
    inp = 512
    assert launch_rules.format_plan(fmt, out, inp, batch).kernel == kernel
    s = gpu.FormatDenseSession(batch, inp, out, gpu.LINEAR, fmt, W=weights(rng, out, inp))
    x = rng.standard_normal((batch, inp)).astype(np.float32)
    x[1:6] *= np.float32(2) ** -np.array([[60], [96], [104], [112], [118]], np.float32)
    x[6] = 0.0
    y, _ = s.execute(x)
    W = s.export_f32().astype(np.float64)
    s.close()
    want = x.astype(np.float64) @ W.T
    assert not y[6].any()
    for r in range(batch):
        if r != 6:
            k = 2.0 ** 126 if 1 <= r < 6 else 1.0
            assert rel_l2(y[r] * k, want[r] * k) <= 2e-6


@pytest.mark.parametrize("fmt", [1, 10])
def test_all_nan_batch_costs_no_recompute(gpu, fmt):
    """A diverged batch, NaN all over, is recomputed to the first NaN of each output
    only: within a few times the clean batch's time (33 times with whole rows)."""
    h = gpu.Hip()
    batch, n = 512, 2048
    s = gpu.FormatDenseSession(batch, n, n, gpu.LINEAR, fmt,
                               blocks=random_blocks(fmt, n, n, np.random.default_rng(fmt)))
    clean = h.upload(np.ones((batch, n), np.float32))
    nan = h.upload(np.full((batch, n), np.nan, np.float32))
    y = h.malloc(batch * n * 4)

    def seconds(x):
        best = 1e9
        for _ in range(20):
            h.sync()
            t = time.perf_counter()
            s.execute_device(x, y, y)
            h.sync()
            best = min(best, time.perf_counter() - t)
        return best

    a, b = seconds(clean), seconds(nan)
    assert np.isnan(h.download(y, (batch, n))).all()
    s.close()
    for p in (clean, nan, y):
        h.free(p)
    assert b <= 4 * a


@pytest.mark.parametrize("batch,kernel,copies", [(1, launch_rules.PER_ROW, 1), (4, launch_rules.PER_ROW, 1),
                                                 (8, launch_rules.ROWS, 2)])
def test_second_copy_of_the_weights_only_where_it_is_read(gpu, batch, kernel, copies):
    """Device memory of four mounted Q4_0 layers of 59 MB of blocks each: twice
    that for a batch of the matrix-core kernels, which read an interleaved copy.
    (The runtime may keep one more freed buffer of that size.)"""
    inp, out, fmt, layers = 32768, 3200, 2, 4
    assert launch_rules.format_plan(fmt, out, inp, batch).kernel == kernel
    h = gpu.Hip()

    def used():
        free, total = ctypes.c_size_t(), ctypes.c_size_t()
        h.sync()
        assert h.h.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return total.value - free.value

    nbytes = inp * out // 32 * 18
    blocks = np.zeros(nbytes, np.uint8)
    mount = lambda: gpu.FormatDenseSession(batch, inp, out, gpu.LINEAR, fmt, blocks=blocks)
    mount().close()  # what the library allocates once
    before = used()
    sessions = [mount() for _ in range(layers)]
    held = used() - before
    for s in sessions:
        s.close()
    assert abs(held / layers - copies * nbytes) < 0.5 * nbytes
