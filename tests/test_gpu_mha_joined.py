"""The joined Q, K and V product of an attention layer: every kernel that can
run it (1 token, 2-4, 5-32, 33 and more with and without a split along K, the
RoPE epilogue and the separate rotation), matrices that do not end on the 128
rows of a tile, every storage, and the layers that are not joined.

Bound: 1e-4 after the attention core, as in the attention layer's other tests
(three-term activations 2e-5 per product).
"""
import numpy as np
import pytest

from test_gpu_dense import rel_l2
from test_gpu_swiglu_mha import oracle_mha

pytestmark = pytest.mark.gpu

CAUSAL, FULL = 1, 2
ROPE, NONE, ALIBI = 0, 1, 2


@pytest.mark.parametrize("dt,scheme", [(16, 3), (4, 2), (5, 1), (4, 3)])
@pytest.mark.parametrize("B,S,H,KVH,hd,mask,pos", [
    (1, 1, 6, 2, 32, CAUSAL, ROPE),     # 192 + 2 x 64 rows, one token
    (1, 1, 32, 8, 128, CAUSAL, ROPE),   # 6144 rows: the matrix-core GEMV where its rule takes it
    (1, 3, 6, 1, 32, CAUSAL, ROPE),     # 192 + 2 x 32
    (2, 2, 5, 1, 64, FULL, NONE),
    (1, 5, 6, 2, 32, CAUSAL, ROPE),     # K ranges and their reduction
    (2, 16, 12, 4, 64, CAUSAL, ROPE),
    (1, 33, 6, 2, 32, CAUSAL, ROPE),    # one row past the small tiles
    (1, 130, 5, 1, 64, CAUSAL, ROPE),   # a ragged second row block; rotated after the product
    (2, 70, 3, 3, 128, FULL, ALIBI),
    (1, 1030, 14, 7, 64, CAUSAL, ROPE),  # 9 x 14 tiles (K split), N % 256 = 0
    (1, 1030, 16, 4, 64, CAUSAL, ROPE),  # 9 x 12 tiles
    (1, 1300, 12, 2, 128, CAUSAL, ROPE),  # 11 x 16 tiles: RoPE in the epilogue
    (2, 650, 12, 4, 96, CAUSAL, ROPE),  # a head width that 128 is no multiple of
    (1, 40, 4, 2, 20, CAUSAL, ROPE),    # 40 K rows: not joined
])
def test_joined_layer_matches_oracle(gpu, oracle, dt, scheme, B, S, H, KVH, hd, mask, pos):
    d = H * hd
    rng = np.random.default_rng(1000 * S + 10 * H + hd + dt)

    def weight(rows, cols):
        return (rng.standard_normal((rows, cols)) / np.sqrt(cols)).astype(np.float32)

    Q, K, V, O = weight(d, d), weight(KVH * hd, d), weight(KVH * hd, d), weight(d, d)
    x = rng.standard_normal((B * S, d)).astype(np.float32)
    s = gpu.MHASession(B, S, d, H, KVH, hd, S, mask, pos, dt, scheme, Q, K, V, O)
    attn, y = s.execute(x)
    s.close()
    oattn, oy = oracle_mha(oracle, dt, scheme, Q, K, V, O, x, B, S, H, KVH, hd, S, mask, pos)
    assert rel_l2(attn, oattn) <= 1e-4
    assert rel_l2(y, oy) <= 1e-4


def test_layer_with_infinite_weight_rows(gpu, oracle):
    """E5M2 rows with infinite codes are recomputed per matrix, not joined: the
    values of that one K/V head are not finite, the others are as without."""
    B, S, H, KVH, hd = 1, 40, 4, 2, 64
    d = H * hd
    rng = np.random.default_rng(7)
    Q, K, V, O = ((rng.standard_normal((n, d)) / np.sqrt(d)).astype(np.float32)
                  for n in (d, KVH * hd, KVH * hd, d))
    V[70, 3] = np.inf  # head 1 of K/V
    x = (np.abs(rng.standard_normal((S, d))) + 0.1).astype(np.float32)
    s = gpu.MHASession(B, S, d, H, KVH, hd, S, CAUSAL, ROPE, 5, 0, Q, K, V, O)
    attn, _ = s.execute(x)
    s.close()
    oattn, _ = oracle_mha(oracle, 5, 0, Q, K, V, O, x, B, S, H, KVH, hd, S, CAUSAL, ROPE)
    assert np.isfinite(oattn).sum() < oattn.size  # the rule keeps the code infinite
    assert np.array_equal(np.isfinite(attn), np.isfinite(oattn))
    ok = np.isfinite(oattn)
    assert rel_l2(attn[ok], oattn[ok]) <= 1e-4
