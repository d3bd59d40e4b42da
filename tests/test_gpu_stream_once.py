"""Kernels that read a large operand once with the non-temporal hint (100 MB and more), and the decode kernel
on head dimensions padded to 64, 128 and 256."""
import numpy as np
import pytest

import tessera_oracle as orc
from tessera_amd import bf16 as b16
from tessera_amd import ops

pytestmark = pytest.mark.gpu
TOL = 2e-3


def _bf(rng, shape):
    return b16.from_float32(rng.standard_normal(shape).astype(np.float32))


# decode shapes at head dimensions off the compiled ones: one and several key splits, a ragged last tile, GQA
# groups of one and two query tiles, several query rows under the causal mask
@pytest.mark.parametrize("D", [16, 48, 80, 112, 144, 240])
@pytest.mark.parametrize("B,Hq,Hkv,Sq,Sk,causal", [(1, 4, 1, 1, 33, False), (2, 8, 2, 4, 1000, True), (3, 4, 4, 1, 4100, False),
                                                   (1, 40, 1, 1, 200, False)])
def test_decode_padded_head_dims(lane, D, B, Hq, Hkv, Sq, Sk, causal):
    rng = np.random.default_rng(D + Sk)
    q, k, v = _bf(rng, (B, Hq, Sq, D)), _bf(rng, (B, Hkv, Sk, D)), _bf(rng, (B, Hkv, Sk, D))
    o, lse = ops.gqa_attention(q, k, v, causal=causal, return_lse=True, out="f32")
    ro, rl = orc.flash_attn_dense(q.to_float32(), k.to_float32(), v.to_float32(), causal=causal)
    assert orc.max_rel_err(o, ro) <= TOL and np.max(np.abs(lse - rl)) <= TOL


# padded head dimensions with as many KV heads as compute units and more: unsplit, two and more rounds, the general kernel
@pytest.mark.parametrize("B,Hq,Hkv,Sk,D", [(32, 8, 8, 513, 80), (37, 8, 8, 300, 96), (33, 8, 8, 1030, 80), (33, 16, 8, 300, 112),
                                           (20, 8, 8, 700, 48), (96, 8, 8, 70, 80)])
def test_decode_padded_many_heads(lane, B, Hq, Hkv, Sk, D):
    rng = np.random.default_rng(B + D)
    q, k, v = _bf(rng, (B, Hq, 1, D)), _bf(rng, (B, Hkv, Sk, D)), _bf(rng, (B, Hkv, Sk, D))
    o, lse = ops.gqa_attention(q, k, v, return_lse=True, out="f32")
    ro, rl = orc.flash_attn_dense(q.to_float32(), k.to_float32(), v.to_float32())
    assert orc.max_rel_err(o, ro) <= TOL and np.max(np.abs(lse - rl)) <= TOL


def test_decode_large_cache(lane):
    B, H, Sk, D = 13, 8, 2051, 128                            # 109 MB of K and V
    rng = np.random.default_rng(1)
    q, k, v = _bf(rng, (B, H, 1, D)), _bf(rng, (B, H, Sk, D)), _bf(rng, (B, H, Sk, D))
    o, lse = ops.gqa_attention(q, k, v, return_lse=True, out="f32")
    ro, rl = orc.flash_attn_dense(q.to_float32(), k.to_float32(), v.to_float32())
    assert orc.max_rel_err(o, ro) <= TOL and np.max(np.abs(lse - rl)) <= TOL


@pytest.mark.parametrize("rows", [5, 100, 1500])              # 128-row tiles; 256-row tiles with 64- and 128-row last ones
def test_grouped_large_weights(lane, rows):
    E, K, N = 8, 1024, 6400                                   # 105 MB of weights
    rng = np.random.default_rng(rows)
    sizes = rng.multinomial(rows, [1 / E] * E)
    off = np.concatenate([[0], np.cumsum(sizes)]).astype(np.int32)
    x, w = _bf(rng, (rows, K)), b16.from_float32((rng.standard_normal((E, K, N)) / 32).astype(np.float32))
    y = ops.grouped_gemm(x, w, group_sizes=sizes, out="f32")
    xf, wf = x.to_float32(), w.to_float32()
    for e in range(E):
        if sizes[e]:
            ref = xf[off[e]:off[e + 1]].astype(np.float64) @ wf[e]
            assert orc.max_rel_err(y[off[e]:off[e + 1]], ref) <= 1e-5
