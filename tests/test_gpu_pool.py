"""The library's memory pool under the resident handles."""
import ctypes
import threading

import numpy as np
import pytest

from tessera_amd import bf16 as b16
from tessera_amd import resident as rs

pytestmark = pytest.mark.gpu


def test_blocks_are_reused_in_default_stream_order(lane):
    lane.load().tessera_gfx950_pool_trim()
    a = lane.PooledBuffer(1000)
    first = a.address
    a.close()
    b = lane.PooledBuffer(1020)                          # the same class
    assert b.address == first
    c = lane.PooledBuffer(1000)
    assert c.address != first                            # still handed out
    assert lane.PooledBuffer(5000).address not in (first, c.address)


def test_shared_blocks_wait_for_a_synchronisation(lane):
    lane.load().tessera_gfx950_pool_trim()
    a = lane.PooledBuffer(3000)
    first = a.ptr                                        # the caller may have work on it in other streams
    a.close()
    b = lane.PooledBuffer(3000)
    assert b.address != first
    lane.synchronize()
    c = lane.PooledBuffer(3000)
    assert c.address == first
    # without one, the pool makes it once 16 of a class wait
    seen = set()
    for _ in range(40):
        x = lane.PooledBuffer(70000)
        seen.add(x.ptr)
        x.close()
    assert len(seen) <= 17


def test_uninitialised_arrays_are_free_of_earlier_work(lane):
    """A new DeviceArray may be written on a stream that nothing orders behind the default one: the products that its memory's
    last owner has queued must not read or overwrite what is written there."""
    hip = ctypes.CDLL("libamdhip64.so", mode=ctypes.RTLD_LOCAL)
    p = ctypes.c_void_p
    hip.hipStreamCreateWithFlags.argtypes = [ctypes.POINTER(p), ctypes.c_uint]
    hip.hipStreamSynchronize.argtypes = hip.hipStreamDestroy.argtypes = [p]
    copy = lane.load().tessera_gfx950_memcpy_d2d_dev
    rng = np.random.default_rng(5)
    n = 4096
    x, w = (rs.DeviceArray.from_host(b16.from_float32((rng.standard_normal((n, n)) / 8).astype(np.float32))) for _ in range(2))
    mine = rs.DeviceArray.from_host(b16.from_float32(np.full((n, n), 3.0, np.float32)))
    want = np.asarray(rs.gemm(rs.gemm(x, w), w).to_host()).view(np.uint16).copy()
    s = p()
    assert hip.hipStreamCreateWithFlags(ctypes.byref(s), 1) == 0          # non-blocking: no order with the default stream
    try:
        for _ in range(10):
            h = rs.gemm(x, w)
            y = rs.gemm(h, w)
            del h
            z = rs.DeviceArray((n, n), "bf16")
            lane.check(copy(z.ptr, mine.ptr, z.nbytes, s), "copy")
            assert hip.hipStreamSynchronize(s) == 0
            assert np.array_equal(np.asarray(y.to_host()).view(np.uint16), want)
            assert np.all(z.to_host().to_float32() == 3.0)
            del y, z
    finally:
        hip.hipStreamDestroy(s)


def test_pool_free_rejects_foreign_addresses(lane):
    lib = lane.load()
    d = lane.DeviceBuffer(64)
    assert lib.tessera_gfx950_pool_free(d.ptr, 0) == lane.BAD_SHAPE
    p = lane.PooledBuffer(64)
    at = p.address
    p.close()
    assert lib.tessera_gfx950_pool_free(at, 0) == lane.BAD_SHAPE         # given back already
    assert lib.tessera_gfx950_pool_free(None, 0) == 0
    assert lib.tessera_gfx950_pool_trim() == 0 and lib.tessera_gfx950_pool_trim() == 0


def test_chains_in_several_threads_keep_their_values(lane):
    """Handles created and dropped by four threads at once: every chain's result is the one it gives alone."""
    rng = np.random.default_rng(3)
    sizes = [64, 96, 128, 160]
    xs = [b16.from_float32(rng.standard_normal((s, 256)).astype(np.float32)) for s in sizes]
    ws = [b16.from_float32((rng.standard_normal((256, 256)) / 16).astype(np.float32)) for _ in range(3)]

    def chain(x):
        h = rs.DeviceArray.from_host(x)
        for w in ws:
            h = rs.gemm(h, rs.DeviceArray.from_host(w))
        return np.asarray(h.to_host()).view(np.uint16)

    want = [chain(x) for x in xs]
    bad = []

    def worker(i):
        for _ in range(20):
            if not np.array_equal(chain(xs[i]), want[i]):
                bad.append(i)

    threads = [threading.Thread(target=worker, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad
