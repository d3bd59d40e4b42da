"""Attention at the sizes where the work is divided differently: workgroups of 128 or 256 query rows and key splits in
the forward, walks shared by several workgroups in the backward.

Bounds: the forward's and backward's of the other attention tests (bf16: probabilities, dS and a stored operand round to
2^-9, f16 to 2^-12; the sums are f32).  One row of 128 or 256 query rows more or less moves the last block, 16 tiles
of 64 keys are the fewest that split, a number of KV heads that is no multiple of 8 changes the order of the grid.
"""
import numpy as np
import pytest

import tessera_oracle as orc
from tessera_amd import bf16, ops

pytestmark = pytest.mark.gpu


def _case(b, hq, hkv, sq, sk, d, dtype, seed=3):
    rng = np.random.default_rng(seed)
    conv = bf16.from_float32 if dtype == "bf16" else (lambda x: x.astype(np.float16))
    back = (lambda x: x.to_float32()) if dtype == "bf16" else (lambda x: x.astype(np.float32))
    t = [conv(rng.standard_normal(s).astype(np.float32)) for s in
         ((b, hq, sq, d), (b, hkv, sk, d), (b, hkv, sk, d), (b, hq, sq, d))]
    return t, [back(x) for x in t]


@pytest.mark.parametrize("b,hq,hkv,sq,sk,d,causal,window,dtype", [
    (1, 2, 1, 127, 127, 128, True, 0, "bf16"), (1, 2, 1, 129, 129, 128, True, 0, "bf16"),
    (2, 8, 4, 257, 257, 64, True, 0, "f16"), (2, 16, 8, 385, 385, 128, True, 0, "bf16"),
    (1, 8, 8, 300, 1030, 128, True, 0, "bf16"), (1, 8, 8, 1024, 1024, 64, False, 0, "f16"),
    (3, 4, 1, 200, 333, 80, True, 0, "bf16"), (2, 8, 8, 300, 300, 48, False, 65, "f16"),
    (1, 16, 8, 512, 1100, 128, True, 70, "bf16"), (1, 4, 4, 700, 300, 64, True, 0, "bf16"),
    (40, 8, 8, 65, 65, 64, True, 0, "bf16"), (1, 8, 1, 140, 3100, 128, True, 0, "f16"),
])
def test_forward_divisions(lane, b, hq, hkv, sq, sk, d, causal, window, dtype):
    (q, k, v, _), (qf, kf, vf, _) = _case(b, hq, hkv, sq, sk, d, dtype)
    kw = {"window": window} if window else {}
    o, lse = ops.gqa_attention(q, k, v, causal=causal, return_lse=True, out="f32", **kw)
    ro, rl = orc.flash_attn_dense(qf, kf, vf, causal=causal, **kw)
    assert orc.max_rel_err(o, ro) <= 2e-3
    seen = np.isfinite(rl)
    assert np.array_equal(np.isfinite(lse), seen) and np.max(np.abs(lse[seen] - rl[seen])) <= 2e-3


@pytest.mark.parametrize("d,causal,sq,sk", [(128, True, 350, 350), (112, False, 290, 400)])
def test_forward_many_heads_past_the_caches(lane, d, causal, sq, sk):
    """K and V of 90 MB in heads that share none: 4-wave workgroups head after head.  Every head and row block must be served by
    its own K and V: reference for the first, the last and a few heads between."""
    b, h = 64, 8
    (q, k, v, _), (qf, kf, vf, _) = _case(b, h, h, sq, sk, d, "bf16")
    o, lse = ops.gqa_attention(q, k, v, causal=causal, return_lse=True, out="f32")
    for i, j in ((0, 0), (0, 7), (1, 0), (31, 3), (40, 5), (63, 7)):
        ro, rl = orc.flash_attn_dense(*(x[i:i + 1, j:j + 1] for x in (qf, kf, vf)), causal=causal)
        assert orc.max_rel_err(o[i, j], ro[0, 0]) <= 2e-3 and np.max(np.abs(lse[i, j] - rl[0, 0])) <= 2e-3, (i, j)


@pytest.mark.parametrize("b,hq,hkv,sq,sk,d,causal,dtype", [
    (1, 8, 1, 512, 512, 128, True, "bf16"),      # 8 heads a group: dK / dV walks shared, heads and tiles split unevenly
    (1, 8, 1, 640, 640, 64, False, "f16"),
    (1, 6, 2, 513, 513, 64, True, "bf16"),       # 3 heads a group, one row past a tile
    (2, 4, 4, 129, 1100, 128, True, "bf16"),     # few query rows, long keys: dQ walks shared
    (1, 4, 1, 1100, 300, 64, True, "f16"),       # more queries than keys
    (1, 2, 2, 1024, 1024, 128, False, "bf16"),
])
def test_backward_shared_walks(lane, b, hq, hkv, sq, sk, d, causal, dtype):
    (q, k, v, do), (qf, kf, vf, dof) = _case(b, hq, hkv, sq, sk, d, dtype, seed=5)
    got = ops.flash_attn_backward(do, q, k, v, causal=causal)
    ref = orc.flash_attn_backward(dof, qf, kf, vf, causal=causal)
    bound = 5e-3 if dtype == "bf16" else 2e-3
    for name, g, r in zip(("dq", "dk", "dv"), got, ref):
        assert orc.max_rel_err(g, r) <= bound, name
    again = ops.flash_attn_backward(do, q, k, v, causal=causal)
    assert all(np.array_equal(x, y) for x, y in zip(got, again))   # sums in split order: the same bits every time
