"""Inputs whose rows keep only the alignment of a float: the split kernel and
the 5-32-row product read them with 16-byte loads moved to the last place that
fits in the row. Widths below one load, around chunks of 128 and around the
padding, rows of an odd stride, and the K ranges of the small product.

Integer inputs and weights whose products and sums are exact in fp32 and on the
matrix cores, so every output is compared exactly; each input row carries its
own values, so a load from a neighbouring row or column shows.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt,scheme", [(4, 2), (16, 3)])
@pytest.mark.parametrize("rows", [5, 16, 17, 32, 33, 130])
@pytest.mark.parametrize("inp", [1, 2, 3, 4, 5, 6, 7, 126, 127, 129, 130, 255, 257, 1023, 2747])
def test_exact_products(gpu, dt, scheme, rows, inp):
    out = 21 if inp != 2747 else 2100
    rng = np.random.default_rng(inp * 100 + rows)
    W = rng.choice(np.float32([-1, 0, 1]), size=(out, inp))
    # a row scale (block exponent) that is a power of two
    W[:, 0] = 240.0 if scheme == 2 else 1.0
    x = rng.integers(-3, 4, size=(rows, inp)).astype(np.float32)
    x[:, -1] = 1 + np.arange(rows) % 3
    s = gpu.DenseSession(rows, inp, out, -1, dt, scheme, W, None)
    pre, _ = s.execute(x)
    s.close()
    assert np.array_equal(pre.astype(np.float64), x.astype(np.float64) @ W.astype(np.float64).T)


@pytest.mark.parametrize("rows", [7, 40])
def test_swiglu_odd_widths(gpu, oracle, rows):
    from test_gpu_dense import rel_l2, tol
    from test_gpu_swiglu_mha import oracle_swiglu

    d, inter = 701, 1303
    rng = np.random.default_rng(rows)
    G, U = ((rng.standard_normal((inter, d)) / np.sqrt(d)).astype(np.float32) for _ in range(2))
    D = (rng.standard_normal((d, inter)) / np.sqrt(inter)).astype(np.float32)
    x = rng.standard_normal((rows, d)).astype(np.float32)
    s = gpu.SwiGLUSession(rows, 1, d, inter, 16, 3, G, U, D)
    h, y = s.execute(x)
    s.close()
    oh, oy = oracle_swiglu(oracle, 16, 3, G, U, D, x)
    assert rel_l2(h, oh) <= tol(rows, 2)
    assert rel_l2(y, oy) <= tol(rows, 3)
