"""Performance cases: the calls a program makes into this library, over the
sizes it makes them at.

Kinds (field "kind" of a case):
  host      a Dense session called with host buffers, as a caller of the C ABI
            calls it (copy in, compute, copy out, wait)
  dense     a Dense session on device buffers: decode (1 row), small batches,
            prefill and projection GEMMs
  swiglu    a SwiGLU feed-forward session on device buffers
  mha       an attention layer: Q, K and V projections, RoPE or ALiBi, masked
            attention, O projection
  volume    the independent cells of a volume, each a chain of Dense layers,
            run as chained groups
  backward  the Dense backward of a training step: d_pre, dX, dW and the loss
  format    a Dense session over ggml block formats mounted from packed blocks

Inputs are made on the GPU from the seed alone. Weights are N(0, 1/in) and
activations N(0, 1), as after a normalisation. Sessions, buffers and the
stream are what a program keeps between calls.
"""
import math
import os
import sys

import numpy as np
import torch

# the binding lives in a folder whose name is no Python package name
sys.path.insert(0, os.path.join(os.getcwd(), "welvet.cuda_amd"))
import pywelvet as pw  # noqa: E402

DTYPES = {"e4m3": pw.E4M3, "e5m2": pw.E5M2, "fp4": pw.FP4}
SCHEMES = {"tensor": pw.SCHEME_TENSOR, "row": pw.SCHEME_ROW, "block32": pw.SCHEME_BLOCK32}
ACTS = {"linear": pw.LINEAR, "relu": pw.RELU, "silu": pw.SILU, "gelu": pw.GELU, "tanh": pw.TANH}
FORMATS = {"q4_0": pw.Q4_0, "q8_0": pw.Q8_0, "q4_k": pw.Q4_K, "q6_k": pw.Q6_K}
FORMAT_BITS = {"q4_0": 4.5, "q8_0": 8.5, "q4_k": 4.5, "q6_k": 6.5625}
MASKS = {"causal": 1, "full": 2}
POSITIONS = {"rope": 0, "none": 1, "alibi": 2, "rope_alibi": 3}


def listed():
    return [
        # A caller of the C ABI with host buffers: the shape the reference
        # quotes its warm execute on (batch 8, 256 -> 256). Latency.
        dict(name="host_256x256_b8", kind="host", rows=8, inp=256, out=256, dtype="e4m3",
             scheme="tensor", act="linear", bias=False),
        # One decode token through a square projection.
        dict(name="dense_4096x4096_e4m3_b1", kind="dense", rows=1, inp=4096, out=4096,
             dtype="e4m3", scheme="row", act="linear", bias=False),
        # A few rows through an odd-sized FP4 layer with bias and activation.
        dict(name="dense_2747x1333_fp4_b7", kind="dense", rows=7, inp=2747, out=1333,
             dtype="fp4", scheme="block32", act="silu", bias=True),
        # Prefill: 4096 tokens through a 1024-wide projection.
        dict(name="dense_1024x1024_e5m2_r4096", kind="dense", rows=4096, inp=1024, out=1024,
             dtype="e5m2", scheme="row", act="linear", bias=False),
        # Feed-forward block, one decode token and a batch of 16 of them.
        dict(name="swiglu_4096x11008_fp4_b1", kind="swiglu", rows=1, inp=4096, inter=11008,
             dtype="fp4", scheme="block32"),
        dict(name="swiglu_4096x11008_fp4_b16", kind="swiglu", rows=16, inp=4096, inter=11008,
             dtype="fp4", scheme="block32"),
        # Attention layer over whole sequences: the benchmark's shape, and
        # ragged sequences with grouped K/V heads and ALiBi.
        dict(name="mha_b8_s512_causal_rope", kind="mha", batch=8, seq=512, heads=16, kv=16, hd=64,
             msl=512, mask="causal", pos="rope", dtype="e5m2", scheme="row"),
        dict(name="mha_b3_s701_gqa_alibi", kind="mha", batch=3, seq=701, heads=12, kv=4, hd=64,
             msl=1024, mask="causal", pos="alibi", dtype="e4m3", scheme="row"),
        # A volume of 64 cells of three 1024-wide layers, batch 256.
        dict(name="volume_64x3x1024_b256", kind="volume", cells=64, layers=3, width=1024, rows=256),
        # Training: the backward of one square layer at a batch of 32, with an
        # MSE target.
        dict(name="backward_4096x4096_b32", kind="backward", rows=32, inp=4096, out=4096,
             dtype="e4m3", scheme="row", act="silu", target=True),
        # Block formats: one decode token, and a prompt of 512 tokens.
        dict(name="q4_k_4096x4096_b1", kind="format", rows=1, inp=4096, out=4096, format="q4_k"),
        dict(name="q8_0_4096x4096_r512", kind="format", rows=512, inp=4096, out=4096,
             format="q8_0"),
    ]


def _log(rng, lo, hi):
    """A whole number from lo to hi, even over the logarithm."""
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _width(rng, lo, hi):
    """A layer width: as often as not a multiple of 64, as model widths are."""
    n = _log(rng, lo, hi)
    return n if rng.random() < 0.4 else max(64, n // 64 * 64)


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        # no dearer than the largest listed case
        if w["flops"] <= 1.0e11 and w["bytes"] <= 1.0e9:
            return c


def _draw(rng):
    kind = rng.choice(["host", "dense", "dense", "dense", "swiglu", "swiglu", "mha", "mha", "mha",
                       "volume", "backward", "backward", "format", "format", "format"])
    if kind == "volume":
        return dict(kind=kind, cells=_log(rng, 2, 64), layers=rng.randint(1, 4),
                    width=rng.choice([256, 384, 512, 768, 1024]), rows=_log(rng, 33, 320))
    if kind == "mha":
        hd = rng.choice([32, 64, 64, 128])
        heads = rng.choice([4, 6, 8, 12, 16])
        kv = rng.choice([k for k in range(1, heads + 1) if heads % k == 0 and heads // k <= 8])
        seq = _log(rng, 1, 1024)
        batch = max(1, min(_log(rng, 1, 16), 4096 // seq))
        msl = max(seq, rng.choice([64, 256, 512, 1024, 2048]))
        return dict(kind=kind, batch=batch, seq=seq, heads=heads, kv=kv, hd=hd, msl=msl,
                    mask=rng.choice(["causal", "causal", "full"]),
                    pos=rng.choice(["rope", "rope", "none", "alibi"]),
                    dtype=rng.choice(sorted(DTYPES)), scheme=rng.choice(["row", "block32"]))
    if kind == "format":
        return dict(kind=kind, rows=_log(rng, 1, 1024), inp=256 * _log(rng, 2, 32),
                    out=_width(rng, 256, 8192), format=rng.choice(sorted(FORMATS)))
    c = dict(kind=kind, dtype=rng.choice(sorted(DTYPES)))
    # FP4 weights are used with block scales, FP8 ones with any
    c["scheme"] = "block32" if c["dtype"] == "fp4" else rng.choice(sorted(SCHEMES))
    if kind == "swiglu":
        c.update(rows=_log(rng, 1, 512), inp=_width(rng, 256, 4096), inter=_width(rng, 512, 11008))
        return c
    c.update(inp=_width(rng, 256, 8192), out=_width(rng, 256, 8192),
             act=rng.choice(["linear", "linear", "relu", "silu", "gelu"]))
    if kind == "backward":
        c.update(rows=_log(rng, 1, 128), target=rng.random() < 0.5)
    else:
        c.update(rows=_log(rng, 1, 64 if kind == "host" else 4096), bias=rng.random() < 0.4)
    return c


# ------------------------------------------------------------------ work ---
def _weight_bytes(n, k, dtype, scheme):
    scales = n * ((k + 31) // 32) if scheme == "block32" else 4 * n
    return n * k * (0.5 if dtype == "fp4" else 1.0) + scales


def work(case):
    k = case["kind"]
    if k in ("host", "dense"):
        m, i, o = case["rows"], case["inp"], case["out"]
        outs = 1 if case["act"] == "linear" and not case["bias"] and k == "dense" else 2
        return {"bytes": _weight_bytes(o, i, case["dtype"], case["scheme"]) + 4 * m * (i + outs * o),
                "flops": 2.0 * m * i * o}
    if k == "swiglu":
        m, i, f = case["rows"], case["inp"], case["inter"]
        w = 2 * _weight_bytes(f, i, case["dtype"], case["scheme"])
        w += _weight_bytes(i, f, case["dtype"], case["scheme"])
        return {"bytes": w + 4 * m * (2 * i + f), "flops": 6.0 * m * i * f}
    if k == "mha":
        t, hd, s = case["batch"] * case["seq"], case["hd"], case["seq"]
        qd, kvd = case["heads"] * hd, case["kv"] * hd
        d = qd
        w = sum(_weight_bytes(n, c, case["dtype"], case["scheme"])
                for n, c in ((qd, d), (kvd, d), (kvd, d), (d, qd)))
        # distinct key rows that a query of batch b can see (the K/V ring
        # holds msl rows)
        keys = sum(s * min((b + 1) * s, case["msl"]) for b in range(case["batch"]))
        return {"bytes": w + 4 * t * (2 * d + qd),
                "flops": 2.0 * t * d * (2 * qd + 2 * kvd) + 4.0 * keys * qd}
    if k == "volume":
        n, m = case["width"], case["rows"]
        w = sum(_weight_bytes(n, n, *_volume_store(j)) for j in range(case["layers"]))
        return {"bytes": case["cells"] * (w + 8.0 * m * n),
                "flops": 2.0 * case["cells"] * case["layers"] * m * n * n}
    if k == "backward":
        m, i, o = case["rows"], case["inp"], case["out"]
        vecs = 3 * m * o + (m * o if case["target"] else 0) + 2 * m * i + i * o
        return {"bytes": _weight_bytes(o, i, case["dtype"], case["scheme"]) + 4.0 * vecs,
                "flops": 4.0 * m * i * o}
    m, i, o = case["rows"], case["inp"], case["out"]
    return {"bytes": i * o * FORMAT_BITS[case["format"]] / 8 + 4.0 * m * (i + o),
            "flops": 2.0 * m * i * o}


def tolerance(case):
    # about four times the distance from exact() that was measured over the
    # listed cases and draws
    k = case["kind"]
    # fp32 activations in three or four low-precision terms on the matrix
    # cores: 2e-5 per product, 4e-5 over the chained ones
    if k in ("host", "dense"):
        return {"rel": 1e-4}
    if k in ("swiglu", "mha", "volume"):
        return {"rel": 2e-4}
    # dX: f64 sums rounded once to f32 (5e-8); dW: rounded to f32 at every
    # batch row, as the reference does (1e-7 at 32 rows)
    if k == "backward":
        return {"rel": 1e-6}
    return {"rel": 2.5e-6}  # fp32 sums of fp32 inputs times exact weights: 2e-7 to 6e-7


# ---------------------------------------------------------------- inputs ---
def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & 0x7FFFFFFFFFFFFFFF)


def _normal(g, *shape, std=1.0):
    return torch.randn(*shape, generator=g, device="cuda", dtype=torch.float32) * std


def _weight(g, out, inp):
    return _normal(g, out, inp, std=1.0 / math.sqrt(inp))


def _host(t):
    return t.cpu().numpy()


def _volume_store(layer):
    """The volume's layers alternate FP8 rows and FP4 blocks."""
    return ("fp4", "block32") if layer % 2 else ("e4m3", "row")


def _inputs(case, seed):
    """Everything that is drawn from the seed, on the GPU."""
    g, k, v = _gen(seed), case["kind"], {}
    if k in ("host", "dense"):
        v["W"] = _weight(g, case["out"], case["inp"])
        v["x"] = _normal(g, case["rows"], case["inp"])
        if case["bias"]:
            v["bias"] = _normal(g, case["out"], std=0.1).double()
    elif k == "swiglu":
        v["G"], v["U"] = (_weight(g, case["inter"], case["inp"]) for _ in range(2))
        v["D"] = _weight(g, case["inp"], case["inter"])
        v["x"] = _normal(g, case["rows"], case["inp"])
    elif k == "mha":
        qd, kvd = case["heads"] * case["hd"], case["kv"] * case["hd"]
        v["Q"], v["K"], v["V"] = _weight(g, qd, qd), _weight(g, kvd, qd), _weight(g, kvd, qd)
        v["O"] = _weight(g, qd, qd)
        v["x"] = _normal(g, case["batch"] * case["seq"], qd)
    elif k == "volume":
        n = case["width"]
        v["W"] = [_weight(g, case["cells"] * n, n).view(case["cells"], n, n)
                  for _ in range(case["layers"])]
        v["x"] = _normal(g, case["cells"], case["rows"], n)
    elif k == "backward":
        m, i, o = case["rows"], case["inp"], case["out"]
        v["W"], v["x"] = _weight(g, o, i), _normal(g, m, i)
        v["pre"] = _normal(g, m, o)
        v["post"] = _act(case["act"], v["pre"].double()).float()
        v["g"] = _normal(g, m, o, std=1.0 if case["target"] else 1.0 / m)
    else:
        W = _weight(g, case["out"], case["inp"])
        v["blocks"], v["W"] = _pack(case["format"], W)
        v["x"] = _normal(g, case["rows"], case["inp"])
    return v


# -------------------------------------------------------- quantised values ---
def _fp8_round(v, mant, bias, top):
    """Nearest FP8 value, ties away from zero; below the least normal: zero."""
    bits = v.abs().contiguous().view(torch.int32)
    field = (bits >> (23 - mant)) - ((127 - bias) << mant) + ((bits >> (22 - mant)) & 1)
    normal = ((bits >> 23) - (127 - bias)) > 0
    mag = ((field << (23 - mant)) + ((127 - bias) << 23)).view(torch.float32).clamp(max=top)
    return torch.where(normal, mag, torch.zeros_like(mag)) * torch.sign(v)


_FP4_MAG = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0)


def _fp4_round(v):
    """Nearest E2M1 value, ties to the smaller magnitude."""
    edges = torch.tensor([(a + b) / 2 for a, b in zip(_FP4_MAG, _FP4_MAG[1:])], device=v.device)
    mags = torch.tensor(_FP4_MAG, device=v.device)
    return mags[torch.bucketize(v.abs(), edges)] * torch.sign(v)


def _dequantised(W, dtype, scheme):
    """W as the library holds it: each element rounded to the dtype under the
    scale scheme, times its scale (a float32 product), widened to float64."""
    maxrep = {"e4m3": 240.0, "e5m2": 57344.0, "fp4": 6.0}[dtype]
    n, k = W.shape
    pad = -k % 32
    if scheme == "block32":
        Wb = torch.nn.functional.pad(W, (0, pad)).view(n, -1, 32)
        amax = Wb.abs().amax(2, keepdim=True)
        f, e = torch.frexp(amax)
        fr, er = math.frexp(maxrep)
        e = torch.where(amax > 0, e - er + (f > fr).int(), torch.zeros_like(e)).double()
        s = torch.exp2(e).float()
        v = Wb / s
    else:
        amax = W.abs().amax() if scheme == "tensor" else W.abs().amax(1, keepdim=True)
        s = (amax.double() / maxrep).float()
        s = torch.where(s == 0, torch.ones_like(s), s)
        v = (W.double() / s.double()).float()
    if dtype == "e4m3":
        q = _fp8_round(v, 3, 7, 448.0)
    elif dtype == "e5m2":
        q = _fp8_round(v, 2, 15, 57344.0)
    else:
        q = _fp4_round(v)
    d = q * s
    return (d.reshape(n, -1)[:, :k] if scheme == "block32" else d).double()


def _f16(t):
    """float16 bytes of a float tensor, and its value."""
    h = t.half()
    return h.contiguous().view(torch.uint8).reshape(*t.shape, 2), h.float()


def _pack(fmt, W):
    """W [out, in] as ggml blocks (uint8 [bytes]) and the float64 weights that
    the blocks stand for."""
    out, inp = W.shape
    u8 = torch.uint8
    if fmt in ("q8_0", "q4_0"):
        b = W.view(-1, 32)
        big = b.gather(1, b.abs().argmax(1, keepdim=True))
        db, d = _f16(big.abs() / 127 if fmt == "q8_0" else big / -8)
        inv = torch.where(d == 0, torch.zeros_like(d), 1 / d)
        if fmt == "q8_0":
            q = torch.round(b * inv).clamp(-127, 127)
            code = q.to(torch.int8).view(u8)
        else:
            q = torch.round(b * inv + 8).clamp(0, 15)
            u = q.to(u8)
            code = u[:, :16] | (u[:, 16:] << 4)
            q = q - 8
        val = q.double() * d.double()
        blocks = torch.cat([db.view(-1, 2), code], 1)
    elif fmt == "q4_k":
        b = W.view(-1, 8, 32)
        lo = b.amin(2).clamp(max=0)
        sc, mn = (b.amax(2).clamp(min=0) - lo) / 15, -lo
        db, d = _f16(sc.amax(1, keepdim=True) / 63)
        mb, dm = _f16(mn.amax(1, keepdim=True) / 63)
        isc = torch.round(sc / d.clamp(min=1e-30)).clamp(0, 63)
        imn = torch.round(mn / dm.clamp(min=1e-30)).clamp(0, 63)
        s, m = (d * isc)[:, :, None], (dm * imn)[:, :, None]
        q = torch.round((b + m) / s.clamp(min=1e-30)).clamp(0, 15)
        val = q.double() * (d.double() * isc.double())[:, :, None]
        val = val - (dm.double() * imn.double())[:, :, None]
        u, a, c = q.to(u8), isc.to(u8), imn.to(u8)
        scales = torch.cat([a[:, :4] | ((a[:, 4:] >> 4) << 6), c[:, :4] | ((c[:, 4:] >> 4) << 6),
                            (a[:, 4:] & 15) | ((c[:, 4:] & 15) << 4)], 1)
        u = u.view(-1, 4, 2, 32)
        code = (u[:, :, 0] | (u[:, :, 1] << 4)).reshape(-1, 128)
        blocks = torch.cat([db.view(-1, 2), mb.view(-1, 2), scales, code], 1)
    else:  # q6_k
        b = W.view(-1, 16, 16)
        sc = b.abs().amax(2) / 31
        db, d = _f16(sc.amax(1, keepdim=True) / 127)
        isc = torch.round(sc / d.clamp(min=1e-30)).clamp(0, 127)
        s = (d * isc)[:, :, None]
        q = torch.round(b / s.clamp(min=1e-30)).clamp(-32, 31)
        val = q.double() * (d.double() * isc.double())[:, :, None]
        u = (q + 32).to(u8).view(-1, 2, 4, 32)  # 128 elements: four rows of 32
        ql = torch.cat([(u[:, :, 0] & 15) | ((u[:, :, 2] & 15) << 4),
                        (u[:, :, 1] & 15) | ((u[:, :, 3] & 15) << 4)], 2).reshape(-1, 128)
        h = u >> 4
        qh = (h[:, :, 0] | (h[:, :, 1] << 2) | (h[:, :, 2] << 4) | (h[:, :, 3] << 6)).reshape(-1, 64)
        blocks = torch.cat([ql, qh, isc.to(torch.int8).view(u8), db.view(-1, 2)], 1)
    return blocks.reshape(-1), val.reshape(out, inp)


# --------------------------------------------------------------- prepare ---
_STREAM = None


def _stream():
    """The one stream that a program queues its passes on."""
    global _STREAM
    if _STREAM is None:
        _STREAM = torch.cuda.Stream()
    return _STREAM.cuda_stream


def prepare(case, seed):
    k, v = case["kind"], _inputs(case, seed)
    st = {"kind": k, "stream": _stream()}

    def empty(*shape, dtype=torch.float32):
        return torch.empty(*shape, device="cuda", dtype=dtype)

    if k in ("host", "dense", "backward"):
        bias = _host(v["bias"]) if "bias" in v else None
        s = pw.DenseSession(case["rows"], case["inp"], case["out"], ACTS[case["act"]],
                            DTYPES[case["dtype"]], SCHEMES[case["scheme"]], _host(v["W"]), bias)
        st["session"] = s
    if k == "host":
        st["x"] = _host(v["x"])
    elif k in ("dense", "format"):
        if k == "format":
            st["session"] = pw.FormatDenseSession(case["rows"], case["inp"], case["out"],
                                                  pw.LINEAR, FORMATS[case["format"]],
                                                  blocks=_host(v["blocks"]))
        st["x"], st["pre"] = v["x"], empty(case["rows"], case["out"])
        plain = k == "format" or (case["act"] == "linear" and not case["bias"])
        st["post"] = st["pre"] if plain else empty(case["rows"], case["out"])
    elif k == "swiglu":
        st["session"] = pw.SwiGLUSession(case["rows"], 1, case["inp"], case["inter"],
                                         DTYPES[case["dtype"]], SCHEMES[case["scheme"]],
                                         *(_host(v[n]) for n in "GUD"))
        st["x"] = v["x"]
        st["pre"], st["post"] = empty(case["rows"], case["inter"]), empty(case["rows"], case["inp"])
    elif k == "mha":
        qd = case["heads"] * case["hd"]
        st["session"] = pw.MHASession(case["batch"], case["seq"], qd, case["heads"], case["kv"],
                                      case["hd"], case["msl"], MASKS[case["mask"]],
                                      POSITIONS[case["pos"]], DTYPES[case["dtype"]],
                                      SCHEMES[case["scheme"]], *(_host(v[n]) for n in "QKVO"))
        t = case["batch"] * case["seq"]
        st["x"], st["pre"], st["post"] = v["x"], empty(t, qd), empty(t, qd)
    elif k == "volume":
        n, m, cells = case["width"], case["rows"], case["cells"]
        acts, groups = [v["x"]], []
        for j in range(case["layers"]):
            dt, sc = _volume_store(j)
            W = _host(v["W"][j])
            sess = [pw.DenseSession(m, n, n, pw.LINEAR, DTYPES[dt], SCHEMES[sc], W[c])
                    for c in range(cells)]
            acts.append(empty(cells, m, n))
            ins, outs = ([t[c].data_ptr() for c in range(cells)] for t in acts[-2:])
            groups.append(pw.DenseGroup(sess, ins, outs, outs))
        # only the last layer's outputs are returned by a volume's cells
        st["chain"] = pw.DenseChain(groups, keep_inner=False)
        st["acts"] = acts
    else:  # backward
        for n in ("x", "pre", "post", "g"):
            st[n] = v[n]
        m, i, o = case["rows"], case["inp"], case["out"]
        st["target"] = case["target"]
        st["dpre"], st["dx"], st["dw"] = empty(m, o), empty(m, i), empty(o, i)
        st["loss"] = empty((m * o + 255) // 256, dtype=torch.float64) if case["target"] else None
    return st


# ------------------------------------------------------------------- run ---
def run(st):
    k, q = st["kind"], st["stream"]
    if k == "host":
        return st["session"].execute(st["x"])
    if k == "volume":
        st["chain"].execute(q)
        return st["acts"][-1]
    if k == "backward":
        loss = st["loss"]
        st["session"].backward_device(
            st["x"].data_ptr(), st["pre"].data_ptr(), st["post"].data_ptr(), st["g"].data_ptr(),
            st["target"], st["dpre"].data_ptr(), st["dx"].data_ptr(), st["dw"].data_ptr(),
            None if loss is None else loss.data_ptr(), q)
        out = [st["dpre"], st["dx"], st["dw"]]
        return out if loss is None else out + [loss]
    pre, post = st["pre"], st["post"]
    st["session"].execute_device(st["x"].data_ptr(), pre.data_ptr(), post.data_ptr(), q)
    return [pre] if post is pre else [pre, post]


# ----------------------------------------------------------------- exact ---
def _act(name, x):
    if name == "relu":
        return x.clamp(min=0)
    if name == "silu":
        return x * torch.sigmoid(x)
    if name == "gelu":
        return 0.5 * x * (1 + torch.tanh(0.7978845608028654 * (x + 0.044715 * x ** 3)))
    if name == "tanh":
        return torch.tanh(x)
    return x


def _act_slope(name, x):
    y = x.clone().requires_grad_(True)
    if name == "linear":
        return torch.ones_like(x)
    return torch.autograd.grad(_act(name, y).sum(), y)[0]


def _exact_mha(case, v):
    b, s, nh, nk, hd = (case[n] for n in ("batch", "seq", "heads", "kv", "hd"))
    t, msl, dev = b * s, case["msl"], "cuda"

    def proj(w, x):
        return x @ _dequantised(w, case["dtype"], case["scheme"]).T

    x = v["x"].double()
    q, k, val = (proj(v[n], x).view(t, -1, hd) for n in "QKV")
    if case["pos"] in ("rope", "rope_alibi"):
        half = hd // 2
        freq = 10000.0 ** (-2.0 * torch.arange(half, device=dev, dtype=torch.float64) / hd)
        ang = torch.arange(t, device=dev, dtype=torch.float64)[:, None, None] * freq
        c, sn = torch.cos(ang), torch.sin(ang)
        q, k = (torch.cat([y[..., :half] * c - y[..., half:] * sn,
                           y[..., :half] * sn + y[..., half:] * c], -1) for y in (q, k))
    k, val = (y.repeat_interleave(nh // nk, 1).transpose(0, 1) for y in (k, val))
    q = q.transpose(0, 1)
    out = torch.empty(nh, t, hd, device=dev, dtype=torch.float64)
    slope = torch.exp2(-8.0 * torch.arange(1, nh + 1, device=dev, dtype=torch.float64) / nh)
    for i in range(b):
        # key positions of all sequences so far, read from a ring of msl rows
        kp = torch.arange((i + 1) * s, device=dev)
        row = (i + 1) * s - 1 - ((i + 1) * s - 1 - kp) % msl
        qp = torch.arange(i * s, (i + 1) * s, device=dev)
        for h in range(nh):
            sc = q[h, qp] @ k[h, row].T / math.sqrt(hd)
            if case["pos"] in ("alibi", "rope_alibi"):
                sc -= slope[h] * (qp[:, None] - kp).abs()
            if case["mask"] == "causal":
                sc.masked_fill_(kp > qp[:, None], -math.inf)
            out[h, qp] = torch.softmax(sc, 1) @ val[h, row]
    attn = out.transpose(0, 1).reshape(t, nh * hd)
    return [attn, proj(v["O"], attn)]


def exact(case, seed):
    k, v = case["kind"], _inputs(case, seed)
    if k == "mha":
        return _exact_mha(case, v)
    if k == "volume":
        x = v["x"].double()
        for j in range(case["layers"]):
            for c in range(case["cells"]):
                x[c] = x[c] @ _dequantised(v["W"][j][c], *_volume_store(j)).T
        return x
    x = v["x"].double()
    if k == "format":
        return [x @ v["W"].T]
    if k == "swiglu":
        def dq(n):
            return _dequantised(v[n], case["dtype"], case["scheme"])

        gate = x @ dq("G").T
        h = gate * torch.sigmoid(gate) * (x @ dq("U").T)
        return [h, h @ dq("D").T]
    W = _dequantised(v["W"], case["dtype"], case["scheme"])
    if k == "backward":
        pre, g = v["pre"].double(), v["g"].double()
        out = []
        if case["target"]:
            d = v["post"].double() - g
            sq = torch.nn.functional.pad((d * d).view(-1), (0, -d.numel() % 256))
            out, g = [sq.view(-1, 256).sum(1)], d * (2.0 / d.numel())
        dpre = g * _act_slope(case["act"], pre)
        return [dpre, dpre @ W, dpre.T @ x] + out
    pre = x @ W.T
    if "bias" in v:
        pre = pre + v["bias"]
    post = _act(case["act"], pre)
    if k == "host":
        return tuple(y.cpu().numpy() for y in (pre, post))
    return [pre] if case["act"] == "linear" and not case["bias"] else [pre, post]
