// Few-row 16-bit GEMM for gfx950: D[M,N] = A[M,K] B[K,N] for up to 64 rows (decode), any N and K.
//
// The product is bound by streaming B from HBM once, so the kernel is built around
// bytes in flight rather than MFMA rate: a workgroup owns a strip of 64 or 128 columns
// of B and a K range, and each of its waves walks its own slices of that range with
// two slices (8 or 16 KB of B per wave) outstanding.  A slice passes through a wave-private LDS
// buffer only to be transposed into MFMA operand order (ds_read_b64_tr_b16); no
// barrier is taken until the waves' partial accumulators are summed through LDS in
// wave order at the end, by all threads at once.  A is read straight from global memory (it is
// small and stays in L2) in operand layout.
//
// LOOSE: the rows of B may lie on any 2-byte boundary (N or the pitch not a multiple of 8, B off a
// 16-byte boundary).  Global memory takes 16-byte loads off their natural alignment, so B is
// still read once, in place, where a copy into an aligned matrix moves it three times.  The
// chunk that straddles the end of a row is loaded from the last eight columns instead, and its lanes
// write the elements that belong to them to LDS one by one.
#pragma once
#include "gemm16.h"
#include "pitch_copy.h"

namespace tsr950 {

// Shape of one wave's work: NJ 32-column blocks (a workgroup owns 32 NJ columns) and
// slices of 32 rows of K.  A slice row is 64 NJ bytes; the LDS row pitch adds 64
// bytes so that the four rows of a transposing read fall in disjoint banks.
template <int NJ>
struct SkinnyShape {
  static constexpr int kCols = 32 * NJ;
  static constexpr int kRows = 32;
  static constexpr int kPitch = 64 * NJ + 64;
  static constexpr int kWaveLds = kRows * kPitch;
  static constexpr int kLoads = 2 * NJ;            // 16-byte loads per lane per slice
  static constexpr int kLanesPerRow = 4 * NJ;
  static constexpr int kRowsPerLoad = 64 / kLanesPerRow;
  static constexpr int kRedPitch = kCols + 4;      // floats per row of a wave's partial tile in LDS
};

// rows: min(M, 32), what one pass of the reduction holds
template <int NW, int NJ>
constexpr int skinny_lds_bytes(int rows) {
  const int slices = NW * SkinnyShape<NJ>::kWaveLds;
  const int sums = NW * rows * SkinnyShape<NJ>::kRedPitch * 4;
  return slices > sums ? slices : sums;
}

// EPI: EPI_F32 or EPI_STORE16.  Split z = blockIdx.y covers K rows [z kps, (z + 1) kps), kps a multiple of 32.
// part != null: the f32 tile of split z goes to part[z][M][gridDim.x kCols] (rows padded to whole
// strips); null: bias, activation and the store to D happen here (one split).
// d_vec: D's rows take vector stores of four elements.
template <class T, int MI, int NW, int NJ, int EPI, bool NT, bool LOOSE>
__global__ __launch_bounds__(NW * 64) void gemm16_skinny_kernel(Gemm16Params p, int kps, float* __restrict__ part, int d_vec) {
  using S = SkinnyShape<NJ>;
  extern __shared__ __align__(16) char smem[];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int l32 = lane & 31, lh = lane >> 5;
  const int n0 = blockIdx.x * S::kCols;
  const int z = blockIdx.y;
  const int kbeg = z * kps;
  const int kend = min(p.K, kbeg + kps);
  const int nslices = kend > kbeg ? (kend - kbeg + S::kRows - 1) / S::kRows : 0;

  // B slice load.  256-byte rows (NJ = 4): a 16-lane write pass is one whole row.
  // 128-byte rows (NJ = 2): the 16-lane groups take rows {0,2},{1,3},{4,6},{5,7} so
  // that one ds_write_b128 pass still covers all 64 banks.
  const int ch = lane % S::kLanesPerRow;
  int brow = lane / S::kLanesPerRow;
  if constexpr (NJ == 2) {
    const int g = lane >> 4, h = (lane >> 3) & 1;
    brow = 4 * (g >> 1) + (g & 1) + 2 * h;
  }
  const int cols_left = p.N - (n0 + ch * 8);           // columns of this lane's chunk inside the row: 8 or more = all
  const bool on = cols_left > 0;
  const bool edge = LOOSE && n0 + S::kCols > p.N && (p.N & 7) != 0;     // some lane's chunk straddles the row's end
  const bool straddle = edge && on && cols_left < 8;
  const int col = LOOSE && cols_left < 8 ? p.N - 8 : n0 + ch * 8;
  uint32_t b_off[S::kLoads];
  uint32_t b_wr[S::kLoads];
#pragma unroll
  for (int q = 0; q < S::kLoads; ++q) {
    const int row = brow + S::kRowsPerLoad * q;
    b_off[q] = on ? (uint32_t)(((long)row * p.ldb + col) * 2) : kOutOfRange;
    b_wr[q] = w * S::kWaveLds + row * S::kPitch + ch * 16;
  }
  // A operand: lane holds row m = 32 mi + l32, k = 16 ks + 8 lh + (0..7).
  uint32_t a_off[MI];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    const int m = mi * 32 + l32;
    a_off[mi] = m < p.M ? (uint32_t)(((long)m * p.lda + 8 * lh) * 2) : kOutOfRange;
  }
  // transposing read: lane supplies k row 8 lh + r16/4 (+4 for the upper half) and
  // columns 32 j + 16 ((lane>>4)&1) + 4 (r16 % 4); it receives column l32, k = 8 lh + (0..7).
  const int r16 = lane & 15;
  const uint32_t b_rd = w * S::kWaveLds + (8 * lh + (r16 >> 2)) * S::kPitch +
                        (16 * ((lane >> 4) & 1) + 4 * (r16 & 3)) * 2;

  f32x16 acc[MI][NJ];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int j = 0; j < NJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mi][j][r] = 0.f;

  uint4 bq[2][S::kLoads], aq[2][2][MI];
  // One slice.  Rows past K are zeros on both sides (the A chunk's eight k are inside K or outside as a
  // whole: the launcher sees to a K or padded copy of A that is a multiple of 8).
  auto load = [&](int slot, int s) __attribute__((always_inline)) {
    const int k0 = kbeg + s * S::kRows;
    const bool whole = k0 + S::kRows <= kend;
    const uint16_t* Bs = p.B + (long)k0 * p.ldb;
    const uint16_t* As = p.A + k0;
#pragma unroll
    for (int q = 0; q < S::kLoads; ++q) {
      const bool in = whole || k0 + brow + S::kRowsPerLoad * q < kend;
      if constexpr (LOOSE) {
        u32x4 v = {0u, 0u, 0u, 0u};
        if (on && in) v = reinterpret_cast<const LooseChunk<uint16_t>*>(reinterpret_cast<const char*>(Bs) + b_off[q])->v;
        bq[slot][q] = make_uint4(v[0], v[1], v[2], v[3]);
      } else {
        bq[slot][q] = buffer_load_b128<NT>(Bs, in ? b_off[q] : kOutOfRange);
      }
    }
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int mi = 0; mi < MI; ++mi)
        aq[slot][ks][mi] = buffer_load_b128(As + ks * 16, whole || k0 + ks * 16 + 8 * lh < kend ? a_off[mi] : kOutOfRange);
  };
  auto consume = [&](int slot, int s_next) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < S::kLoads; ++q) {
      if (!straddle) lds_write_b128(smem, b_wr[q], bq[slot][q]);
    }
    if (edge && straddle) {
      // element e of the loaded chunk is column N - 8 + e: the last cols_left of them are this lane's
#pragma unroll
      for (int q = 0; q < S::kLoads; ++q) {
        const uint32_t wd[4] = {bq[slot][q].x, bq[slot][q].y, bq[slot][q].z, bq[slot][q].w};
#pragma unroll
        for (int e = 1; e < 8; ++e)
          if (e >= 8 - cols_left)
            *reinterpret_cast<uint16_t*>(smem + b_wr[q] + (e - (8 - cols_left)) * 2) = (uint16_t)(wd[e >> 1] >> (16 * (e & 1)));
      }
    }
    uint4 af[2][MI];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int mi = 0; mi < MI; ++mi) af[ks][mi] = aq[slot][ks][mi];
    // (the transposing read returns elements other lanes wrote: nothing may move across this point)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    uint4 bf[2][NJ];
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int j = 0; j < NJ; ++j) {
        const char* pb = smem + b_rd + ks * 16 * S::kPitch + j * 64;
        const uint2 lo = lds_read_tr16_b64(pb);
        const uint2 hi = lds_read_tr16_b64(pb + 4 * S::kPitch);
        bf[ks][j] = make_uint4(lo.x, lo.y, hi.x, hi.y);
      }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    if (s_next < nslices) load(slot, s_next);
#pragma unroll
    for (int ks = 0; ks < 2; ++ks)
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int mi = 0; mi < MI; ++mi) acc[mi][j] = mfma_32x32x16<T>(bf[ks][j], af[ks][mi], acc[mi][j]);
  };

  int s = w;
  if (s < nslices) load(0, s);
  if (s + NW < nslices) load(1, s + NW);
  for (; s + NW < nslices; s += 2 * NW) {
    consume(0, s + 2 * NW);
    consume(1, s + 3 * NW);
  }
  if (s < nslices) consume(0, nslices);

  // ---- sum the waves' partial tiles: every wave puts the rows that exist into LDS, then all threads
  // add the NW copies of four columns in wave order and store them ----
  // acc[mi][j][r]: row m = 32 mi + l32, col n = n0 + 32 j + 8 (r/4) + 4 lh + (r%4).
  float* red = reinterpret_cast<float*>(smem);
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    const int rows = min(p.M - mi * 32, 32);
    if (rows <= 0) break;
    __syncthreads();                                   // slices consumed / the last pass read
    if (l32 < rows) {
      float* dst = red + ((long)w * rows + l32) * S::kRedPitch + lh * 4;
#pragma unroll
      for (int j = 0; j < NJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q)
          *reinterpret_cast<float4*>(dst + j * 32 + q * 8) = make_float4(acc[mi][j][4 * q], acc[mi][j][4 * q + 1],
                                                                        acc[mi][j][4 * q + 2], acc[mi][j][4 * q + 3]);
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < rows * (S::kCols / 4); idx += NW * 64) {
      const int row = idx / (S::kCols / 4), c = idx % (S::kCols / 4) * 4;
      float4 v = *reinterpret_cast<const float4*>(red + (long)row * S::kRedPitch + c);
#pragma unroll
      for (int u = 1; u < NW; ++u) {
        const float4 x = *reinterpret_cast<const float4*>(red + ((long)u * rows + row) * S::kRedPitch + c);
        v.x += x.x; v.y += x.y; v.z += x.z; v.w += x.w;
      }
      const int m = mi * 32 + row;
      if (part) {
        *reinterpret_cast<float4*>(part + ((long)z * p.M + m) * ((long)gridDim.x * S::kCols) + n0 + c) = v;
        continue;
      }
      store_quad<T, EPI>(p.D, (long)m * p.ldd, n0 + c, p.N, v, p.bias, p.act, d_vec);
    }
  }
}

}  // namespace tsr950
