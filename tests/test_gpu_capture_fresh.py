"""Calls that use the stream's workspace where it is there, recorded on a stream that has run nothing and has none."""
import ctypes

import numpy as np
import pytest

import tessera_oracle as orc
from tessera_amd import bf16 as b16

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def hip():
    L = ctypes.CDLL("libamdhip64.so", mode=ctypes.RTLD_LOCAL)
    p, pp = ctypes.c_void_p, ctypes.POINTER(ctypes.c_void_p)
    for name, args in {"hipStreamCreate": [pp], "hipStreamSynchronize": [p], "hipStreamDestroy": [p],
                       "hipStreamBeginCapture": [p, ctypes.c_int], "hipStreamEndCapture": [p, pp],
                       "hipGraphInstantiate": [pp, p, p, p, ctypes.c_size_t], "hipGraphLaunch": [p, p],
                       "hipGraphExecDestroy": [p], "hipGraphDestroy": [p]}.items():
        getattr(L, name).argtypes = args
    return L


def _bits(rng, shape):
    return np.asarray(b16.from_float32(rng.standard_normal(shape).astype(np.float32)), np.uint16)


def _gemm16(lane, rng, M, N, K):
    a, b = _bits(rng, (M, K)), _bits(rng, (K, N))
    ref = b16.from_bits(a).to_float32().astype(np.float64) @ b16.from_bits(b).to_float32()
    d = [lane.DeviceBuffer.from_host(x) for x in (a, b)] + [lane.DeviceBuffer(M * N * 4)]
    fn = lane.load().tessera_gfx950_gemm_bf16_dev
    return d, (lambda s: fn(d[0].ptr, d[1].ptr, d[2].ptr, M, N, K, s)), ref, np.float32, 1e-5   # f32 sums


def _gemm8(lane, rng, M, N, K, fp8):
    a, b = (rng.integers(0, 120, s).astype(np.uint8) for s in ((M, K), (K, N)))
    d = [lane.DeviceBuffer.from_host(x) for x in (a, b)] + [lane.DeviceBuffer(M * N * 4)]
    lib = lane.load()
    if fp8:
        fn = lib.tessera_gfx950_gemm_e4m3_f32_dev
        one = ctypes.c_float(1.0)
        return (d, (lambda s: fn(d[0].ptr, d[1].ptr, one, one, d[2].ptr, M, N, K, s)), orc.gemm_fp8_codes(a, b, 1.0, 1.0),
                np.float32, 1e-5)
    fn = lib.tessera_gfx950_gemm_i8_i32_dev
    return d, (lambda s: fn(d[0].ptr, d[1].ptr, d[2].ptr, M, N, K, s)), orc.gemm_i8_i32(a.view(np.int8), b.view(np.int8)), np.int32, 0


def _attention(lane, rng, B, Hq, Hkv, Sq, Sk, D):
    q, k, v = _bits(rng, (B, Hq, Sq, D)), _bits(rng, (B, Hkv, Sk, D)), _bits(rng, (B, Hkv, Sk, D))
    ref, _ = orc.flash_attn_dense(*(b16.from_bits(x).to_float32() for x in (q, k, v)))
    d = [lane.DeviceBuffer.from_host(x) for x in (q, k, v)] + [lane.DeviceBuffer(q.size * 4)]
    fn = lane.load().tessera_gfx950_flash_attn_gqa_bf16_dev
    return (d, (lambda s: fn(*(x.ptr for x in d), None, B, Hq, Hkv, Sq, Sk, D, ctypes.c_float(D ** -0.5), 0, 0, s)), ref,
            np.float32, 2e-3)                                 # probabilities round to 2^-9


CASES = {
    "gemm_copy_of_a": lambda lane, rng: _gemm16(lane, rng, 5, 131, 777),       # K off 8: A would be copied
    "gemm_split": lambda lane, rng: _gemm16(lane, rng, 33, 1003, 1024),        # N off 8: only the K split needs scratch
    "gemm_strips": lambda lane, rng: _gemm16(lane, rng, 27, 3520, 5312),       # on the grid, few rows on tiles
    "gemm_strips_9": lambda lane, rng: _gemm16(lane, rng, 9, 3520, 5312),      # on the grid, 128-column strips
    "gemm_tiles_split": lambda lane, rng: _gemm16(lane, rng, 150, 576, 5384),  # tiles, K in eight parts that are not equal
    "int8_copy_of_a": lambda lane, rng: _gemm8(lane, rng, 5, 131, 777, False),
    "int8_on_the_grid": lambda lane, rng: _gemm8(lane, rng, 16, 512, 1024, False),
    "fp8_split": lambda lane, rng: _gemm8(lane, rng, 5, 131, 1024, True),
    "decode_padded": lambda lane, rng: _attention(lane, rng, 24, 8, 8, 1, 1500, 80),
    "decode_padded_split": lambda lane, rng: _attention(lane, rng, 4, 8, 8, 1, 900, 80),
}


@pytest.mark.parametrize("case", CASES)
def test_records_without_a_workspace(lane, hip, case):
    _record_and_replay(lane, hip, *CASES[case](lane, np.random.default_rng(len(case))))


@pytest.mark.parametrize("case", ["gemm_strips_9", "gemm_tiles_split"])
def test_records_beside_a_smaller_workspace(lane, hip, case):
    """The stream has the workspace of a smaller eager call (1 MiB, the smallest; these need 1.1 and 2.8 MB)."""
    from tessera_amd.schedule import select_gfx950_gemm_schedule as sel
    assert sel(9, 3520, 5312).workgroup_tile == (32, 128, 32) and 9 * 3520 * 4 * sel(9, 3520, 5312).split_k > 1 << 20
    assert sel(150, 576, 5384).workgroup_tile[0] == 64 and 150 * 576 * 4 * sel(150, 576, 5384).split_k > 1 << 20
    rng = np.random.default_rng(len(case))
    small, run_small, *_ = _gemm16(lane, rng, 5, 131, 777)
    try:
        _record_and_replay(lane, hip, *CASES[case](lane, rng), before=run_small)
    finally:
        for x in small:
            x.close()


def _record_and_replay(lane, hip, d, enqueue, ref, dtype, tol, before=None):
    lane.load().tessera_gfx950_probe()
    s, graph, exe = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_void_p()
    assert hip.hipStreamCreate(ctypes.byref(s)) == 0
    lane.load().tessera_gfx950_stream_release(s)               # (a handle that an earlier test's stream had)
    try:
        if before:
            assert before(s) == 0 and hip.hipStreamSynchronize(s) == 0
        assert hip.hipStreamBeginCapture(s, 0) == 0
        rc = enqueue(s)
        ended = hip.hipStreamEndCapture(s, ctypes.byref(graph))
        assert rc == 0 and ended == 0 and graph.value
        assert hip.hipGraphInstantiate(ctypes.byref(exe), graph, None, None, 0) == 0
        for replay in range(3):
            d[-1].zero()
            lane.synchronize()
            assert hip.hipGraphLaunch(exe, s) == 0 and hip.hipStreamSynchronize(s) == 0
            got = d[-1].download(ref.shape, dtype)
            assert orc.max_rel_err(got, ref) <= tol if tol else np.array_equal(got, ref), replay
            assert enqueue(None) == 0                         # eager work between the replays, with a workspace
            lane.synchronize()
            got = d[-1].download(ref.shape, dtype)
            assert orc.max_rel_err(got, ref) <= tol if tol else np.array_equal(got, ref), replay
    finally:
        if exe.value:
            hip.hipGraphExecDestroy(exe)
        if graph.value:
            hip.hipGraphDestroy(graph)
        hip.hipStreamSynchronize(s)
        hip.hipStreamDestroy(s)
        for x in d:
            x.close()
