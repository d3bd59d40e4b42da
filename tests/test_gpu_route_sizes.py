"""Routing at the sizes where its launch plan changes: one workgroup for everything (up to 16 tokens), for the plan
(up to 6144 slots), the three-pass form above; expert counts either side of 64, 128 and 256; k past one wave."""
import numpy as np
import pytest

import tessera_oracle as orc
from tessera_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T,E,k,cap", [(1, 1, 1, 0), (16, 64, 8, 0), (16, 65, 3, 2), (17, 8, 8, 0), (15, 1024, 70, 0), (768, 8, 8, 0),
                                       (769, 8, 8, 300), (2048, 129, 3, 0), (2049, 300, 3, 20), (6145, 7, 1, 0), (97, 64, 64, 33),
                                       (8192, 256, 8, 100), (700, 1000, 9, 0)])
@pytest.mark.parametrize("ties", [False, True])
def test_route_sizes(lane, T, E, k, cap, ties):
    rng = np.random.default_rng(T + E + k)
    lg = rng.standard_normal((T, E)).astype(np.float32)
    if ties:
        lg = np.round(lg * 2) / 2                        # many equal logits: the lowest expert wins
    lib = lane.load()
    S = T * k
    d = lane.DeviceBuffer.from_host(lg)
    tos, eos, cw, gs, go, n = (lane.DeviceBuffer(4 * max(m, 4)) for m in (S, S, S, E, E + 1, 1))
    lane.check(lib.tessera_gfx950_moe_route_f32_dev(d.ptr, T, E, k, 1, cap, tos.ptr, eos.ptr, cw.ptr, gs.ptr, go.ptr, n.ptr, None),
               "route")
    lane.synchronize()
    # the definition, in numpy: softmax, stable descending order, first come first kept, stable sort by expert
    p = np.exp(lg - lg.max(1, keepdims=True))
    p = (p / p.sum(1, keepdims=True, dtype=np.float32)).astype(np.float32)
    order = np.argsort(-lg, axis=1, kind="stable")[:, :k]
    flat = order.reshape(-1)
    rank = np.zeros(S, np.int64)
    seen = np.zeros(E, np.int64)
    for s, e in enumerate(flat):
        rank[s] = seen[e]
        seen[e] += 1
    keep = rank < (cap if cap else S + 1)
    slots = np.flatnonzero(keep)
    slots = slots[np.argsort(flat[slots], kind="stable")]
    m = len(slots)
    assert int(n.download((1,), np.int32)[0]) == m
    assert np.array_equal(tos.download((S,), np.int32)[:m], slots // k)
    assert np.array_equal(eos.download((S,), np.int32)[:m], flat[slots])
    sizes = np.bincount(flat[slots], minlength=E)
    assert np.array_equal(gs.download((E,), np.int32), sizes)
    assert np.array_equal(go.download((E + 1,), np.int32), np.concatenate([[0], np.cumsum(sizes)]))
    w = np.take_along_axis(p, order, 1)
    w = w / w.sum(1, keepdims=True) if k > 1 else w
    # exp to two units, sums of up to 1024 terms and two divisions
    assert np.max(np.abs(cw.download((S,), np.float32)[:m] - w.reshape(-1)[slots])) <= 2e-6
