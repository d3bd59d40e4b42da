"""The few-row streaming kernels (16-bit and 8-bit): rows of B on and off the 16-byte grid, K that no slice
divides, strips that end inside a chunk, one and two row blocks."""
import numpy as np
import pytest

import tessera_oracle as orc
from tessera_amd import bf16 as b16
from tessera_amd import ops

pytestmark = pytest.mark.gpu

# M up to 8 / 32 / 64; N below, at and past a strip of 128, off 8 and off 16; K below a slice, off 8, off 32, split
EDGES = [(1, 8, 1), (1, 9, 33), (3, 127, 31), (8, 129, 257), (9, 128, 256), (16, 1003, 771), (17, 136, 300), (31, 384, 2056),
         (32, 2054, 3391), (32, 8200, 1030), (33, 250, 515), (63, 1001, 1500), (64, 515, 520), (16, 12352, 4104)]


@pytest.mark.parametrize("M,N,K", EDGES)
@pytest.mark.parametrize("st", ["bf16", "f16"])
def test_few_rows_16bit(lane, M, N, K, st):
    rng = np.random.default_rng(M * 1000 + N + K)
    A = rng.standard_normal((M, K)).astype(np.float32)
    B = (rng.standard_normal((K, N)) / np.sqrt(K)).astype(np.float32)
    a = b16.from_float32(A) if st == "bf16" else A.astype(np.float16)
    b = b16.from_float32(B) if st == "bf16" else B.astype(np.float16)
    ref = orc.gemm_f64(A, B, st)
    got = ops.gemm(a, b, out="f32")
    assert orc.max_rel_err(got, ref) <= 1e-5                              # f32 sums of up to 4104 products
    assert np.array_equal(ops.gemm(a, b, out="f32"), got)                 # fixed summation order
    stored = ops.gemm(a, b)
    sf = stored.to_float32() if st == "bf16" else stored.astype(np.float32)
    assert np.array_equal(sf, orc.round_to_storage(got, st))
    bias = rng.standard_normal(N).astype(np.float32)
    fused = ops.fused_gemm(a, b, bias=bias, activation="relu")
    assert orc.max_rel_err(fused, np.maximum(ref + bias, 0.0)) <= 1e-5


@pytest.mark.parametrize("M,N,K", [(1, 16, 1), (1, 17, 65), (8, 129, 2049), (16, 4808, 1600), (31, 250, 130), (32, 128, 64),
                                   (33, 1003, 771), (64, 1030, 4097), (20, 6336, 1280), (64, 272, 2112)])
def test_few_rows_8bit(lane, M, N, K):
    rng = np.random.default_rng(M + N + K)
    xq = rng.integers(-127, 128, (M, K)).astype(np.int8)
    wq = rng.integers(-127, 128, (K, N)).astype(np.int8)
    acc = orc.gemm_i8_i32(xq, wq)
    assert np.array_equal(ops.gemm_i8(xq, wq), acc)
    rs, cs = rng.random((M, 1)).astype(np.float32), rng.random(N).astype(np.float32)
    y, got_acc = ops.w8a8_gemm(xq, wq, rs, cs, return_acc=True)
    assert np.array_equal(got_acc, acc)
    assert np.array_equal(y, (acc.astype(np.float32) * rs) * cs)
    codes_a, _, sa = orc.quantize_fp8_e4m3(rng.standard_normal((M, K)).astype(np.float32))
    codes_b, _, sb = orc.quantize_fp8_e4m3(rng.standard_normal((K, N)).astype(np.float32))
    assert orc.max_rel_err(ops.gemm_fp8(codes_a, codes_b, sa, sb, out="f32"), orc.gemm_e4m3(codes_a, codes_b, sa, sb)) <= 2e-3


# up to 32 rows off the 16-byte grid: one slice of K for each of eight waves (8-bit: K 512) and beyond, whole, last and
# missing slices of four waves, unsplit and split K
@pytest.mark.parametrize("M,N,K", [(16, 1003, 512), (16, 1003, 513), (32, 2055, 577), (9, 141, 1025), (31, 4099, 1301), (24, 131, 4100)])
def test_few_rows_off_the_grid_in_four_waves(lane, M, N, K):
    rng = np.random.default_rng(M + N + K)
    a, b = rng.integers(-127, 128, (M, K)).astype(np.int8), rng.integers(-127, 128, (K, N)).astype(np.int8)
    assert np.array_equal(ops.gemm_i8(a, b), orc.gemm_i8_i32(a, b))
    A, B = rng.standard_normal((M, K)).astype(np.float32), (rng.standard_normal((K, N)) / np.sqrt(K)).astype(np.float32)
    got = ops.gemm(b16.from_float32(A), b16.from_float32(B), out="f32")
    assert orc.max_rel_err(got, orc.gemm_f64(A, B, "bf16")) <= 1e-5      # f32 sums of up to 4100 products


# fp8 off the 16-byte grid, below 2^24 multiply-adds or under 16 rows (one and two row blocks, split and unsplit K)
@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
@pytest.mark.parametrize("M,N,K", [(1, 17, 203), (5, 130, 201), (15, 1003, 2111), (33, 33, 203), (64, 1003, 259)])
def test_few_rows_fp8_adds_small_products(lane, fmt, M, N, K):
    """Products 14 binary places below their neighbours: every partial sum has at most 21 bits, so sums in f32 are exact
    in any order, where the fp8 matrix instruction drops all of them (4e-4 of the result)."""
    big, small = (0x58, 0x20) if fmt == "e4m3" else (0x4C, 0x30)          # 16 and 1/8
    at = np.arange(K) % 8 == 3
    a = np.where(at, big, small).astype(np.uint8) * np.ones((M, 1), np.uint8)
    b = (np.where(at, big, small).astype(np.uint8) * np.ones((N, 1), np.uint8)).T
    want = at.sum() * 256.0 + (~at).sum() / 64.0
    assert want * 64 < 2 ** 24
    got = ops.gemm_fp8(a, np.ascontiguousarray(b), 1.0, 1.0, out="f32", format=fmt)
    assert np.all(got == want), np.unique(got)[:5]


@pytest.mark.parametrize("fmt", ["e4m3", "e5m2"])
def test_few_rows_fp8_every_code(lane, fmt):
    """All 256 codes times one, in an off-grid product of 16 rows: the value itself; a column that
    holds an infinity or a NaN is NaN throughout."""
    one = 0x38 if fmt == "e4m3" else 0x3C
    a = np.where(np.eye(16, dtype=bool), one, 0).astype(np.uint8)
    b = np.zeros((16, 17), np.uint8)
    b[:, :16] = np.arange(256, dtype=np.uint8).reshape(16, 16).T          # column n: codes 16 n .. 16 n + 15
    table = (orc.e4m3_decode_table() if fmt == "e4m3" else orc.e5m2_decode_table()).astype(np.float64)
    with np.errstate(invalid="ignore"):
        want = table[a] @ table[b]
    got = ops.gemm_fp8(a, b, 1.0, 1.0, out="f32", format=fmt)
    assert np.array_equal(got, want.astype(np.float32), equal_nan=True)
