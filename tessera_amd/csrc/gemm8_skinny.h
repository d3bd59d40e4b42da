// Skinny 8-bit GEMM for gfx950: raw accumulators of D[M,N] = A[M,K] B[K,N] for M <= 64
// (quantised decode: a few activation rows against a big int8 / e4m3 weight matrix).
//
// The product is bound by streaming B from HBM once.  A workgroup of G8S_NW waves owns a strip of
// 128 columns of B and a K range; each of its waves walks its own 64-row slices of that range with two
// slices (16 KB of B per wave) outstanding.  A slice passes through a wave-private LDS buffer
// only to be transposed into MFMA operand order (ds_read_b64_tr_b8), no barrier is taken until
// the waves' partial accumulators are summed through LDS in wave order at the end, by all threads at once, and
// A is read straight from global memory in operand layout (it is small and stays in L2).
// With K split over workgroups the raw accumulators (int32, or f32 of unscaled e4m3 products) of split
// z = blockIdx.y are summed by gemm8_split_sum_kernel; unsplit, the epilogue runs here.
#pragma once
#include "gemm8.h"
#include "pitch_copy.h"

namespace tsr950 {

constexpr int G8S_NJ = 4;                       // 32-column blocks per strip
constexpr int G8S_COLS = 32 * G8S_NJ;           // 128
constexpr int G8S_ROWS = 64;                    // k rows per slice
constexpr int G8S_PITCH = G8S_COLS + 32;        // the pad spreads the 8 rows of a transposing read over all banks
constexpr int G8S_WAVE_LDS = G8S_ROWS * G8S_PITCH;
constexpr int G8S_LOADS = G8S_ROWS * G8S_COLS / 16 / 64;     // 16-byte loads per lane per slice: 8
constexpr int G8S_RED_PITCH = G8S_COLS + 4;     // words per row of a wave's partial tile in LDS
// LDS of a workgroup of NW waves: the waves' slices (10 KB each), then reused by one pass of the
// reduction (`rows` = min(M, 32) rows of every wave's partial tile)
constexpr int g8s_smem(int nw, int rows) {
  return nw * G8S_WAVE_LDS > nw * rows * G8S_RED_PITCH * 4 ? nw * G8S_WAVE_LDS : nw * rows * G8S_RED_PITCH * 4;
}

// Eight fp8 codes as bf16, which holds every e4m3 and e5m2 value exactly.
template <class T>
__device__ __forceinline__ uint4 widen8_f8(uint32_t lo, uint32_t hi) {
  auto pair = [](uint32_t w, auto upper) __attribute__((always_inline)) {
    constexpr bool U = decltype(upper)::value;
    if constexpr (std::is_same<T, BF8>::value) return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_bf8(w, 1.f, U));
    else return __builtin_bit_cast(uint32_t, __builtin_amdgcn_cvt_scalef32_pk_bf16_fp8(w, 1.f, U));
  };
  return make_uint4(pair(lo, std::false_type{}), pair(lo, std::true_type{}), pair(hi, std::false_type{}), pair(hi, std::true_type{}));
}

// LOOSE: rows of B on any byte boundary, as in the 16-bit kernel (gemm16_skinny.h); A then comes in rows
// of lda bytes padded with zeros to a multiple of 16.
// WIDEN (fp8): the codes are multiplied as bf16.  The fp8 matrix instruction drops products more than 13 binary
// places below the largest of their run of 8; the one-thread-per-element kernel, in whose place this form stands,
// adds every product in f32, and so do the bf16 instructions.  The conversions and four times the matrix
// instructions cost up to a tenth (64 x 100 x 1001 17.5 -> 18.9 us, 5 x 8191 x 1001 38.5 -> 42.7; element by
// element 301 and 395).
// part: the raw accumulators of split z go to part[z][M][strips * 128]; null (one split): through the
// product's epilogue to D.
template <class T, int G8S_NW, int MI, int EPI, bool LOOSE, bool WIDEN>
__global__ __launch_bounds__(G8S_NW * 64) void gemm8_skinny_kernel(const Gemm8Params p, int lda, int kps, void* __restrict__ part,
                                                                   int vec) {
  const uint8_t* A = p.A;
  const uint8_t* B = p.B;
  const int M = p.M, N = p.N, K = p.K;
  constexpr bool IS_I8 = std::is_same<T, I8>::value;
  using acc_t = typename std::conditional<IS_I8, i32x16, f32x16>::type;
  extern __shared__ __align__(16) char smem[];
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  const int l32 = lane & 31, lh = lane >> 5;
  const int n0 = blockIdx.x * G8S_COLS;
  const int z = blockIdx.y;
  const int kbeg = z * kps;
  const int kend = min(K, kbeg + kps);
  const int nslices = kend > kbeg ? (kend - kbeg + G8S_ROWS - 1) / G8S_ROWS : 0;

  // B slice load: 8 lanes cover one 128-byte row, one load instruction 8 rows.
  const int ch = lane & 7, brow = lane >> 3;
  const int cols_left = N - (n0 + ch * 16);            // columns of this lane's chunk inside the row: 16 or more = all
  const bool on = cols_left > 0;
  const bool edge = LOOSE && n0 + G8S_COLS > N && (N & 15) != 0;        // some lane's chunk straddles the row's end
  const bool straddle = edge && on && cols_left < 16;
  const int col = LOOSE && cols_left < 16 ? N - 16 : n0 + ch * 16;
  uint32_t b_off[G8S_LOADS], b_wr[G8S_LOADS];
#pragma unroll
  for (int q = 0; q < G8S_LOADS; ++q) {
    const int row = brow + 8 * q;
    b_off[q] = on ? (uint32_t)row * (uint32_t)N + col : kOutOfRange;
    b_wr[q] = w * G8S_WAVE_LDS + row * G8S_PITCH + ch * 16;
  }
  // A operand: lane holds row m = 32 mi + l32, bytes k = 32 f + 16 lh + (0..15) of the slice.
  uint32_t a_off[MI];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
    a_off[mi] = 32 * mi + l32 < M ? (uint32_t)(32 * mi + l32) * (uint32_t)lda + 16 * lh : kOutOfRange;
  // transposing read: lane r of a 16-lane block supplies row k0 + r/2 and columns 8 (r%2) .. +7 of a
  // 16-column patch; lane i receives column i, k0 .. k0 + 7.
  const int r16 = lane & 15;
  const uint32_t b_rd = w * G8S_WAVE_LDS + (16 * lh + (r16 >> 1)) * G8S_PITCH + 16 * ((lane >> 4) & 1) + 8 * (r16 & 1);

  acc_t acc[MI][G8S_NJ];
#pragma unroll
  for (int mi = 0; mi < MI; ++mi)
#pragma unroll
    for (int j = 0; j < G8S_NJ; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) acc[mi][j][r] = 0;

  uint4 bq[2][G8S_LOADS], aq[2][MI][2];
  // One slice.  Rows past K are zeros on both sides (a lane's sixteen k of A are inside K or outside as a
  // whole, or zeros in the padded copy).
  auto load = [&](int slot, int s) __attribute__((always_inline)) {
    const int k0 = kbeg + s * G8S_ROWS;
    const bool whole = k0 + G8S_ROWS <= kend;
    const uint8_t* Bs = B + (long)k0 * N;
    const uint8_t* As = A + k0;
#pragma unroll
    for (int q = 0; q < G8S_LOADS; ++q) {
      const bool in = whole || k0 + brow + 8 * q < kend;
      if constexpr (LOOSE) {
        u32x4 v = {0u, 0u, 0u, 0u};
        if (on && in) v = reinterpret_cast<const LooseChunk<uint8_t>*>(Bs + b_off[q])->v;
        bq[slot][q] = make_uint4(v[0], v[1], v[2], v[3]);
      } else {
        bq[slot][q] = buffer_load_b128(Bs, in ? b_off[q] : kOutOfRange);
      }
    }
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) {
      aq[slot][mi][0] = buffer_load_b128(As, whole || k0 + 16 * lh < kend ? a_off[mi] : kOutOfRange);
      aq[slot][mi][1] = buffer_load_b128(As + 32, whole || k0 + 32 + 16 * lh < kend ? a_off[mi] : kOutOfRange);
    }
  };
  auto consume = [&](int slot, int s_next) __attribute__((always_inline)) {
#pragma unroll
    for (int q = 0; q < G8S_LOADS; ++q) {
      if (!straddle) lds_write_b128(smem, b_wr[q], bq[slot][q]);
    }
    if (edge && straddle) {
      // byte e of the loaded chunk is column N - 16 + e: the last cols_left of them are this lane's
#pragma unroll
      for (int q = 0; q < G8S_LOADS; ++q) {
        const uint32_t wd[4] = {bq[slot][q].x, bq[slot][q].y, bq[slot][q].z, bq[slot][q].w};
#pragma unroll
        for (int e = 1; e < 16; ++e)
          if (e >= 16 - cols_left) *reinterpret_cast<uint8_t*>(smem + b_wr[q] + e - (16 - cols_left)) = (uint8_t)(wd[e >> 2] >> (8 * (e & 3)));
      }
    }
    uint4 af[MI][2];
#pragma unroll
    for (int mi = 0; mi < MI; ++mi) { af[mi][0] = aq[slot][mi][0]; af[mi][1] = aq[slot][mi][1]; }
    // (the transposing read returns bytes other lanes wrote: nothing may move across this point)
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    uint4 bf[2][G8S_NJ];
#pragma unroll
    for (int f = 0; f < 2; ++f)
#pragma unroll
      for (int j = 0; j < G8S_NJ; ++j) {
        const char* pb = smem + b_rd + f * 32 * G8S_PITCH + j * 32;
        const uint2 lo = lds_read_tr8_b64(pb);
        const uint2 hi = lds_read_tr8_b64(pb + 8 * G8S_PITCH);
        bf[f][j] = make_uint4(lo.x, lo.y, hi.x, hi.y);
      }
    asm volatile("" ::: "memory");
    __builtin_amdgcn_wave_barrier();
    if (s_next < nslices) load(slot, s_next);
    if constexpr (WIDEN && !IS_I8) {
      // (8 bytes of a lane: the same eight k of A and B, whichever they are)
#pragma unroll
      for (int f = 0; f < 2; ++f)
#pragma unroll
        for (int h = 0; h < 2; ++h) {
          uint4 aw[MI];
#pragma unroll
          for (int mi = 0; mi < MI; ++mi)
            aw[mi] = h ? widen8_f8<T>(af[mi][f].z, af[mi][f].w) : widen8_f8<T>(af[mi][f].x, af[mi][f].y);
#pragma unroll
          for (int j = 0; j < G8S_NJ; ++j) {
            const uint4 bw = h ? widen8_f8<T>(bf[f][j].z, bf[f][j].w) : widen8_f8<T>(bf[f][j].x, bf[f][j].y);
#pragma unroll
            for (int mi = 0; mi < MI; ++mi) acc[mi][j] = mfma_32x32x16<BF16>(bw, aw[mi], acc[mi][j]);
          }
        }
      return;
    }
#pragma unroll
    for (int mi = 0; mi < MI; ++mi)
#pragma unroll
      for (int j = 0; j < G8S_NJ; ++j) {
        if constexpr (IS_I8) {
          acc[mi][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, bf[0][j]),
                                                             __builtin_bit_cast(i32x4, af[mi][0]), acc[mi][j], 0, 0, 0);
          acc[mi][j] = __builtin_amdgcn_mfma_i32_32x32x32_i8(__builtin_bit_cast(i32x4, bf[1][j]),
                                                             __builtin_bit_cast(i32x4, af[mi][1]), acc[mi][j], 0, 0, 0);
        } else {
          const i32x4 b0 = __builtin_bit_cast(i32x4, bf[0][j]), b1 = __builtin_bit_cast(i32x4, bf[1][j]);
          const i32x4 x0 = __builtin_bit_cast(i32x4, af[mi][0]), x1 = __builtin_bit_cast(i32x4, af[mi][1]);
          const i32x8 b8 = (i32x8){b0[0], b0[1], b0[2], b0[3], b1[0], b1[1], b1[2], b1[3]};
          const i32x8 a8 = (i32x8){x0[0], x0[1], x0[2], x0[3], x1[0], x1[1], x1[2], x1[3]};
          acc[mi][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(b8, a8, acc[mi][j], f8_format<T>(), f8_format<T>(),
                                                                       0, 0, 0, 0);
        }
      }
  };

  int s = w;
  if (s < nslices) load(0, s);
  if (s + G8S_NW < nslices) load(1, s + G8S_NW);
  for (; s + G8S_NW < nslices; s += 2 * G8S_NW) {
    consume(0, s + 2 * G8S_NW);
    consume(1, s + 3 * G8S_NW);
  }
  if (s < nslices) consume(0, nslices);

  // ---- sum the waves' partial tiles: every wave puts the rows that exist into LDS, then all threads add
  // the copies of four columns in wave order and store them; rows of a split's tile are padded to whole strips ----
  // acc[mi][j][r]: row m = 32 mi + l32, column n0 + 32 j + 8 (r / 4) + 4 lh + (r % 4): runs of four columns
  using elem_t = g8_elem<T>;
  using quad_t = g8_quad<T>;
  elem_t* red = reinterpret_cast<elem_t*>(smem);
  elem_t* out = reinterpret_cast<elem_t*>(part) + (size_t)z * M * gridDim.x * G8S_COLS;
#pragma unroll
  for (int mi = 0; mi < MI; ++mi) {
    const int rows = min(M - mi * 32, 32);
    if (rows <= 0) break;
    __syncthreads();                                   // slices consumed / the last pass read
    if (l32 < rows) {
      elem_t* dst = red + ((long)w * rows + l32) * G8S_RED_PITCH + lh * 4;
#pragma unroll
      for (int j = 0; j < G8S_NJ; ++j)
#pragma unroll
        for (int q = 0; q < 4; ++q) {
          const quad_t v = {acc[mi][j][4 * q], acc[mi][j][4 * q + 1], acc[mi][j][4 * q + 2], acc[mi][j][4 * q + 3]};
          *reinterpret_cast<quad_t*>(dst + j * 32 + q * 8) = v;
        }
    }
    __syncthreads();
    for (int idx = threadIdx.x; idx < rows * (G8S_COLS / 4); idx += G8S_NW * 64) {
      const int row = idx / (G8S_COLS / 4), c = idx % (G8S_COLS / 4) * 4;
      quad_t v = *reinterpret_cast<const quad_t*>(red + (long)row * G8S_RED_PITCH + c);
#pragma unroll
      for (int u = 1; u < G8S_NW; ++u) v += *reinterpret_cast<const quad_t*>(red + ((long)u * rows + row) * G8S_RED_PITCH + c);
      if (!part) gemm8_store_quad<T, EPI>(p, mi * 32 + row, n0 + c, v, vec);
      else *reinterpret_cast<quad_t*>(out + (size_t)(mi * 32 + row) * gridDim.x * G8S_COLS + n0 + c) = v;
    }
  }
}

}  // namespace tsr950
