"""dX and dW of batches on the f64 matrix cores and the 8-row outer product, at
the edges of their tiles: 16 batch rows, 256 columns, 16 code rows per unit, 8
waves, with one band of code rows (dX written directly) and with several.

Integer inputs: every product and partial sum is exact in f64 and its result
in f32, so dX is bit-exact in any order; dW follows the reference's rounding at
every batch row and is bit-exact always."""
import numpy as np
import pytest

from test_gpu_dense import rel_l2

pytestmark = pytest.mark.gpu


def run(gpu, oracle, dt, scheme, batch, inp, out, act, target, x, W, pre, g):
    h = gpu.Hip()
    s = gpu.DenseSession(batch, inp, out, act, dt, scheme, W)
    post = np.array([[oracle.activate(act, float(v)) for v in r] for r in pre], np.float32)
    n = batch * out
    bufs = {k: h.upload(v) for k, v in dict(x=x, pre=pre, post=post, g=g).items()}
    sizes = dict(dpre=4 * n, dx=4 * batch * inp, dw=4 * out * inp, loss=8 * ((n + 255) // 256))
    bufs.update({k: h.malloc(v) for k, v in sizes.items()})
    for _ in range(2):  # the second on used buffers
        s.backward_device(bufs["x"], bufs["pre"], bufs["post"], bufs["g"], target, bufs["dpre"],
                          bufs["dx"], bufs["dw"], bufs["loss"])
    h.sync()
    got = [h.download(bufs["dpre"], (batch, out)), h.download(bufs["dx"], (batch, inp)),
           h.download(bufs["dw"], (out, inp))]
    Wd = s.export_f32()
    s.close()
    for p in bufs.values():
        h.free(p)
    return got, Wd


SHAPES = [
    (3, 32, 7),       # fewer code rows than a unit, one tile mostly padding
    (16, 256, 128),   # exactly one tile and group
    (17, 257, 130),   # one past each
    (33, 1000, 1500), # several bands, ragged columns and rows
    (64, 300, 40),    # more groups than code rows per wave
    (130, 520, 144),
    (5, 4100, 260),
    (300, 2100, 33),  # as many workgroups as CUs without bands
]


@pytest.mark.parametrize("dt,scheme", [(4, 2), (4, 3), (5, 1), (5, 3), (16, 3), (16, 2)])
@pytest.mark.parametrize("batch,inp,out", SHAPES)
def test_batched_backward_exact_on_integers(gpu, oracle, dt, scheme, batch, inp, out):
    rng = np.random.default_rng(dt * 100 + scheme * 10 + batch)
    W = rng.integers(-2, 3, (out, inp)).astype(np.float32)
    x = rng.integers(-4, 5, (batch, inp)).astype(np.float32)
    g = rng.integers(-4, 5, (batch, out)).astype(np.float32)
    pre = rng.standard_normal((batch, out)).astype(np.float32)
    (dpre, dx, dw), Wd = run(gpu, oracle, dt, scheme, batch, inp, out, -1, False, x, W, pre, g)
    assert np.array_equal(dpre, g)
    # weights that the scheme does not hold exactly still give exact f64 terms
    want = g.astype(np.float64) @ Wd.astype(np.float64)
    if np.array_equal(Wd, W):
        assert np.array_equal(dx, want.astype(np.float32))
    else:
        assert rel_l2(dx, want) <= 1e-6
    assert np.array_equal(dw, (g.T.astype(np.float64) @ x).astype(np.float32))


@pytest.mark.parametrize("batch,inp,out", [(3, 100, 50), (18, 600, 333), (40, 513, 258)])
@pytest.mark.parametrize("act,target", [(-1, False), (0, True), (1, True), (2, False)])
def test_batched_backward_matches_oracle(gpu, oracle, batch, inp, out, act, target):
    rng = np.random.default_rng(batch + inp + act)
    W = (rng.standard_normal((out, inp)) / np.sqrt(inp)).astype(np.float32)
    x, pre, g = (rng.standard_normal(s).astype(np.float32)
                 for s in ((batch, inp), (batch, out), (batch, out)))
    (dpre, dx, dw), Wd = run(gpu, oracle, 4, 2, batch, inp, out, act, target, x, W, pre, g)
    # from the d_pre that was returned: dW bit for bit, dX to one f32 rounding
    _, odx, odw = oracle.backward(Wd, dpre, pre, x, -1)
    assert np.array_equal(dw, odw)
    assert rel_l2(dx, odx) <= 1e-7


def test_batched_backward_keeps_non_finite_rows_apart(gpu, oracle):
    """An infinite gradient of one batch row stays in that row of dX."""
    rng = np.random.default_rng(3)
    batch, inp, out = 20, 300, 200
    W = rng.standard_normal((out, inp)).astype(np.float32)
    x, pre, g = (rng.standard_normal(s).astype(np.float32)
                 for s in ((batch, inp), (batch, out), (batch, out)))
    (_, clean, _), _ = run(gpu, oracle, 4, 2, batch, inp, out, -1, False, x, W, pre, g)
    g[7, 5], g[18, 6] = np.inf, np.nan
    (_, dx, _), Wd = run(gpu, oracle, 4, 2, batch, inp, out, -1, False, x, W, pre, g)
    keep = [b for b in range(batch) if b not in (7, 18)]
    assert np.array_equal(dx[keep], clean[keep])
    with np.errstate(invalid="ignore"):
        want = g[7].astype(np.float64) @ Wd.astype(np.float64)
    assert np.array_equal(np.isnan(dx[7]), np.isnan(want)) and np.isnan(dx[18]).all()
