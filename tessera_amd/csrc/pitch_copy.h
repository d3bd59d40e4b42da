// Copies between a matrix of any pitch and alignment and a 16-byte aligned, zero-padded one:
// how operands that the 16-byte loads of the tile kernels cannot take reach those kernels.
#pragma once
#include <algorithm>
#include "common.h"
#include "pad_blocks.h"

namespace tsr950 {

// A thread moves one 16-byte chunk: threadIdx.x runs along a row, threadIdx.y over rows; the copy back has its blocks along
// a row, over rows and over the batch in blockIdx.x, y and z, the padding copy all of them along x (pad_blocks.h).  The side of
// any alignment is accessed with one 16-byte instruction where the whole chunk is inside the row (global memory takes accesses off
// their natural alignment), element by element at the row's end.
// (the field is a plain vector type: a packed attribute is ignored on a field of class type, which would
// leave the struct 16-byte aligned and the access free to assume it)
template <class E> struct __attribute__((packed, aligned(sizeof(E)))) LooseChunk { u32x4 v; };
static_assert(alignof(LooseChunk<uint8_t>) == 1 && alignof(LooseChunk<uint16_t>) == 2 && sizeof(LooseChunk<uint16_t>) == 16,
              "LooseChunk must carry its element's alignment");

// dst[b][r][c] (rows_dst x ld_dst, 16-byte aligned) = src[b][r][c] inside rows_src x cols_src, else 0.
template <class E> struct PadJob {
  E* dst;
  long ld_dst, stride_dst;
  const E* src;
  long ld_src, stride_src;
  int rows_src, cols_src, rows_dst;
  int batch = 0;                         // filled in by PadLaunch, as are its blocks and the launch's blocks up to here
  PadBlocks blocks{};
  unsigned end = 0;
};
// Up to three matrices in one launch (the operands of a product and a vector that goes with them, as bytes of E): each launch
// more costs a small product 3 to 5 us (int8 1017 x 734 x 2905 45.6 us in a launch each, 35.0 in one).  The jobs' blocks lie
// one after the other along blockIdx.x: on a common grid of the widest and the tallest job most blocks were empty (int8 74 x
// 557 x 11705 65 us, 34 so).
template <class E> struct PadJobs { PadJob<E> job[kPadJobs]; };
// The rows r0, r0 + step, ... of product b, this thread's 16-byte chunk of each.
template <class E>
__device__ __forceinline__ void pad_rows(const PadJob<E>& j, long b, long c0, int r0, int step) {
  constexpr int V = 16 / sizeof(E);
  for (int r = r0; r < j.rows_dst; r += step) {
    uint4 out = make_uint4(0u, 0u, 0u, 0u);
    if (r < j.rows_src && c0 < j.cols_src) {
      const E* sp = j.src + b * j.stride_src + (long)r * j.ld_src + c0;
      if (c0 + V <= j.cols_src) {
        const u32x4 t = reinterpret_cast<const LooseChunk<E>*>(sp)->v;
        out = make_uint4(t[0], t[1], t[2], t[3]);
      } else {
        alignas(16) E v[V];
#pragma unroll
        for (int u = 0; u < V; ++u) v[u] = c0 + u < j.cols_src ? sp[u] : E(0);
        out = *reinterpret_cast<const uint4*>(v);
      }
    }
    *reinterpret_cast<uint4*>(j.dst + b * j.stride_dst + (long)r * j.ld_dst + c0) = out;
  }
}
template <class E>
__global__ void __launch_bounds__(64 * kCopyRowsPerBlock) pad_rows_kernel(const PadJobs<E> jobs) {
  const unsigned id = blockIdx.x;
  const int which = id < jobs.job[0].end ? 0 : id < jobs.job[1].end ? 1 : 2;
  const PadJob<E>& j = jobs.job[which];
  const unsigned at = id - (which ? jobs.job[which - 1].end : 0u), bx = j.blocks.bx, by = j.blocks.by, per = bx * by;
  const unsigned b0 = at / per, in = at - b0 * per;
  const long c0 = ((long)(in % bx) * 64 + threadIdx.x) * (16 / sizeof(E));
  if (c0 >= j.ld_dst) return;
  for (long b = b0; b < j.batch; b += j.blocks.bz)
    pad_rows(j, b, c0, (int)(in / bx) * kCopyRowsPerBlock + threadIdx.y, (int)by * kCopyRowsPerBlock);
}
// One matrix of one product, a few rows of A in front of a streaming product as a rule: blocks along a row in blockIdx.x, over
// the rows in y, without the choice of a job and the two divisions in front of the first load.  (60 products of up to 64 rows in 16 bits, off the
// grid: 0.7 % less time than through the kernel above; 120 in 8 bits 0.1 %.)
template <class E>
__global__ void __launch_bounds__(64 * kCopyRowsPerBlock) pad_one_kernel(const PadJob<E> j) {
  const long c0 = ((long)blockIdx.x * 64 + threadIdx.x) * (16 / sizeof(E));
  if (c0 >= j.ld_dst) return;
  pad_rows(j, 0, c0, blockIdx.y * kCopyRowsPerBlock + threadIdx.y, gridDim.y * kCopyRowsPerBlock);
}
// dst[b][r][c] = src[b][r][c] for r < rows, c < cols; src 16-byte aligned with pitch ld_src, dst any.
template <class E>
__global__ void __launch_bounds__(64 * kCopyRowsPerBlock)
unpad_rows_kernel(E* __restrict__ dst, long ld_dst, long stride_dst, const E* __restrict__ src, long ld_src,
                  long stride_src, int rows, int cols) {
  constexpr int V = 16 / sizeof(E);
  const int c0 = (blockIdx.x * 64 + threadIdx.x) * V;
  if (c0 >= cols) return;
  const long b = blockIdx.z;
  for (int r = blockIdx.y * kCopyRowsPerBlock + threadIdx.y; r < rows; r += gridDim.y * kCopyRowsPerBlock) {
    const uint4 in = *reinterpret_cast<const uint4*>(src + b * stride_src + (long)r * ld_src + c0);
    E* dp = dst + b * stride_dst + (long)r * ld_dst + c0;
    if (c0 + V <= cols) {
      reinterpret_cast<LooseChunk<E>*>(dp)->v = u32x4{in.x, in.y, in.z, in.w};
    } else {
      alignas(16) E v[V];
      *reinterpret_cast<uint4*>(v) = in;
#pragma unroll
      for (int u = 0; u < V; ++u)
        if (c0 + u < cols) dp[u] = v[u];
    }
  }
}
inline dim3 copy_grid(long rows, long ld, int vec, int batch) {
  const long bx = (ld / vec + 63) / 64, by = (rows + kCopyRowsPerBlock - 1) / kCopyRowsPerBlock;
  return dim3((unsigned)bx, (unsigned)std::max<long>(1, std::min<long>(by, 16384)), (unsigned)batch);
}
inline dim3 copy_block() { return dim3(64, kCopyRowsPerBlock, 1); }

// Collects the jobs of one launch.
template <class E>
class PadLaunch {
 public:
  explicit PadLaunch(int batch) : batch_(batch) {}
  void add(PadJob<E> j) { push(j, batch_); }
  // a vector of n 4-byte values, padded to n_dst (whose bytes are a multiple of 16)
  void add_vector(float* dst, long n_dst, const float* src, int n) {
    constexpr int per = 4 / sizeof(E);
    push({reinterpret_cast<E*>(dst), n_dst * per, 0, reinterpret_cast<const E*>(src), (long)n * per, 0, 1, n * per, 1}, 1);
  }
  void run(hipStream_t s) const {
    const PadJob<E>& j = jobs_.job[0];
    if (count_ == 1 && j.batch == 1)
      hipLaunchKernelGGL(pad_one_kernel<E>, dim3(j.blocks.bx, j.blocks.by), copy_block(), 0, s, j);
    else if (count_)
      hipLaunchKernelGGL(pad_rows_kernel<E>, dim3(jobs_.job[count_ - 1].end), copy_block(), 0, s, jobs_);
  }

 private:
  void push(PadJob<E> j, int batch) {
    j.batch = batch;
    j.blocks = pad_blocks(j.rows_dst, j.ld_dst, 16 / sizeof(E), batch);
    j.end = (count_ ? jobs_.job[count_ - 1].end : 0u) + j.blocks.bx * j.blocks.by * j.blocks.bz;
    jobs_.job[count_++] = j;
  }
  PadJobs<E> jobs_{};
  int batch_, count_ = 0;
};

}  // namespace tsr950
