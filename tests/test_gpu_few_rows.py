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
