"""Matrix-core attention over every mask and position kind: the window and
prefix masks, ALiBi, short rings and the sigmoid, at the edges of its tiles
(64 or 32 keys), of its workgroups (64, 128 or 256 queries) and of the K/V
ring, against the f64 oracle.

Q, K and V are signed permutations (times a power of two) and the inputs
multiples of 1/4 up to 2, so the projections are exact and the comparison is
of the attention alone. Bound: the scores of up to a few tens, the exponents
and the sums are fp32 (2^-24 relative each, about 1e-6 over a few hundred
keys); without GEN operands of two bf16 terms leave 2^-16 per product.
"""
import numpy as np
import pytest

import cxx_probe
from test_gpu_dense import rel_l2

pytestmark = pytest.mark.gpu

CAUSAL, FULL, WINDOW, PREFIX = 1, 2, 3, 4
ROPE, NONE, ALIBI, ROPE_ALIBI = 0, 1, 2, 3


def signed_permutation(rng, rows, cols, scale):
    """rows <= cols: every output is one input, signed and scaled."""
    W = np.zeros((rows, cols), np.float32)
    W[np.arange(rows), rng.permutation(cols)[:rows]] = rng.choice([-scale, scale], rows)
    return W


def layer(seed, B, S, H, KVH, hd):
    rng = np.random.default_rng(seed)
    d = H * hd
    Q = signed_permutation(rng, d, d, 0.5)
    K = signed_permutation(rng, KVH * hd, d, 1.0)
    V = signed_permutation(rng, KVH * hd, d, 1.0)
    O = signed_permutation(rng, d, d, 1.0)
    x = (rng.integers(-8, 9, size=(B * S, d)) / 4).astype(np.float32)
    return Q, K, V, O, x


@pytest.mark.parametrize("B,S,H,KVH,hd,msl,mask,pos,window,wc,prefix,sig", [
    (1, 1, 2, 1, 64, 64, CAUSAL, ALIBI, 0, 1, 0, 0),        # one query, one key
    (2, 16, 4, 2, 64, 16, CAUSAL, ALIBI, 0, 1, 0, 0),       # ring of one tile's quarter
    (3, 65, 3, 3, 32, 65, CAUSAL, ALIBI, 0, 1, 0, 0),       # one key past a tile
    (3, 70, 3, 1, 128, 80, FULL, ALIBI, 0, 1, 0, 0),        # rows above the query, ring wraps
    (4, 50, 2, 2, 64, 64, FULL, ROPE_ALIBI, 0, 1, 0, 0),
    (2, 300, 40, 8, 64, 300, CAUSAL, ALIBI, 0, 1, 0, 0),    # 8-wave workgroups at hd 64
    (4, 256, 64, 8, 64, 512, CAUSAL, ALIBI, 0, 1, 0, 0),    # the widest, output split written
    (2, 200, 70, 7, 32, 256, CAUSAL, ROPE_ALIBI, 0, 1, 0, 0),
    (2, 129, 64, 64, 128, 200, CAUSAL, ALIBI, 0, 1, 0, 0),  # 8 waves at hd 128
    (3, 100, 2, 2, 64, 128, WINDOW, ROPE, 17, 1, 0, 0),     # window of its own and the past batch
    (3, 100, 2, 2, 64, 128, WINDOW, NONE, 33, 0, 0, 0),     # both sides
    (3, 100, 2, 2, 32, 100, WINDOW, ALIBI, 250, 0, 0, 0),   # wider than the ring
    (2, 90, 2, 1, 64, 100, PREFIX, NONE, 0, 1, 40, 0),
    (2, 90, 2, 1, 128, 100, PREFIX, ALIBI, 0, 1, 130, 0),   # prefix into the second sequence
    (5, 20, 2, 2, 64, 20, CAUSAL, NONE, 0, 1, 0, 0),        # ring shorter than a tile
    (5, 20, 2, 2, 64, 24, FULL, ROPE, 0, 1, 0, 0),
    (3, 40, 2, 2, 64, 48, WINDOW, NONE, 30, 1, 0, 1),       # sigmoid weights
    (3, 40, 2, 2, 32, 48, CAUSAL, ALIBI, 0, 1, 0, 1),       # sigmoid with ALiBi: per position
    (2, 33, 4, 2, 64, 64, CAUSAL, NONE, 0, 1, 0, 0),        # narrow workgroups, plain masks
    (2, 200, 20, 4, 64, 256, FULL, NONE, 0, 1, 0, 0),
    (1, 100, 3, 3, 128, 128, CAUSAL, NONE, 0, 1, 0, 0),
])
def test_attention_matches_oracle(gpu, oracle, B, S, H, KVH, hd, msl, mask, pos, window, wc, prefix,
                                  sig):
    Q, K, V, O, x = layer(B * 1000 + S + hd + mask, B, S, H, KVH, hd)
    d = H * hd
    attn, y = cxx_probe.mha_masked(B, S, d, H, KVH, msl, mask, pos, window, wc, prefix, sig, 4, Q,
                                   K, V, O, x)
    q, k, v = x @ Q.T, x @ K.T, x @ V.T
    want = oracle.mha_attention(q, k, v, B, S, H, KVH, hd, msl, mask, pos, sig, window, prefix,
                                1 if mask == CAUSAL else wc, threads=8)
    plain = mask in (CAUSAL, FULL) and pos in (ROPE, NONE) and msl >= 64
    err = rel_l2(attn, want)
    print(f"attention B={B} S={S} H={H} hd={hd} mask={mask} pos={pos}: rel-L2 {err:.2e}")
    assert err <= (2e-5 if plain else 3e-6)
    # the O projection reads the attention output that was returned
    assert rel_l2(y, attn @ O.T) <= 5e-5


@pytest.mark.parametrize("bad", [np.inf, -np.inf])  # (the FP6 input split turns NaN finite)
@pytest.mark.parametrize("hd,msl", [(64, 128), (32, 100), (128, 300)])
def test_non_finite_token_stays_with_the_queries_that_see_it(gpu, oracle, bad, hd, msl):
    """One token whose V is not finite: the queries before it (causal, one
    sequence) are those of the clean input, the others are not finite where
    the oracle's are not."""
    B, S, H, d = 1, 100, 2, 2 * hd
    Q, K, V, O, x = layer(hd, B, S, H, H, hd)
    t = 70
    V = V.copy()
    col = int(np.flatnonzero(V[5])[0])
    Q[:, col] = 0.0  # the value reaches V alone
    K[:, col] = 0.0
    xb = x.copy()
    xb[t, col] = bad
    attn, _ = cxx_probe.mha_masked(B, S, d, H, H, msl, CAUSAL, ALIBI, 0, 1, 0, 0, 4, Q, K, V, O, xb)
    clean, _ = cxx_probe.mha_masked(B, S, d, H, H, msl, CAUSAL, ALIBI, 0, 1, 0, 0, 4, Q, K, V, O, x)
    assert np.isfinite(attn[:t]).all()
    assert rel_l2(attn[:t], clean[:t]) <= 3e-6
    assert not np.isfinite(attn[t:, 5]).any()


@pytest.mark.parametrize("B,S,msl", [(40, 1, 1), (64, 1, 2), (40, 2, 2), (40, 3, 4), (60, 4, 4),
                                     (30, 8, 8), (20, 15, 15), (20, 16, 16)])
@pytest.mark.parametrize("H,hd", [(1, 64), (2, 32), (1, 128)])
@pytest.mark.parametrize("mask", [CAUSAL, FULL])
def test_short_alibi_rings_keep_their_digits(gpu, oracle, B, S, msl, H, hd, mask):
    """Rings of a few rows that each stand for many positions, under the flattest
    slopes (2^-8, with two heads also 2^-4): the sum over a row's positions is
    r^c - 1 over r - 1 with r near 1. Inputs of +-1, so an output's error is that of
    the weights. Bound: exponents of a few units rounded to f32 (2^-24 of 4 is
    2.4e-7) and weights of 2^-23, together 3.6e-7 of weights that sum to 1; with 1 - r
    formed in f32 it was 2e-6."""
    rng = np.random.default_rng(B + S + hd)
    Q, K, V, O, _ = layer(B + hd, B, S, H, H, hd)
    d = H * hd
    x = rng.choice(np.float32([-1, 1]), size=(B * S, d))
    attn, _ = cxx_probe.mha_masked(B, S, d, H, H, msl, mask, ALIBI, 0, 1, 0, 0, 4, Q, K, V, O, x)
    want = oracle.mha_attention(x @ Q.T, x @ K.T, x @ V.T, B, S, H, H, hd, msl, mask, ALIBI, 0, 0, 0,
                                1, threads=8)
    err = float(np.max(np.abs(attn - want)))
    print(f"ring of {msl}, {B} x {S}, {H} x {hd}: largest error {err:.2e}")
    assert err <= 3.6e-7
