// How a launch that copies up to three matrices divides into blocks (host code, no device headers).
#pragma once
#include <algorithm>

namespace tsr950 {

constexpr int kCopyRowsPerBlock = 4;
constexpr int kPadJobs = 3;
// HIP takes fewer than 2^32 threads along x, with 64 to a block fewer than 2^26 blocks: a quarter of that for each
// of three matrices.
constexpr long kPadJobBlocks = 1L << 24;

// bx blocks along a row, by over the rows, bz over the batch.  Rows and products beyond by and bz are walked in strides
// by the blocks there are; a row is always covered (its bytes in 16-byte chunks, 64 to a block, are under 2^24 blocks).
struct PadBlocks { unsigned bx, by, bz; };
inline PadBlocks pad_blocks(long rows, long ld, int vec, long batch) {
  const long bx = std::max(1L, (ld / vec + 63) / 64), most = std::max(1L, kPadJobBlocks / bx);
  const long bz = std::min(batch, most);
  const long by = std::min((rows + kCopyRowsPerBlock - 1) / kCopyRowsPerBlock, std::min(16384L, most / bz));
  return {(unsigned)bx, (unsigned)std::max(1L, by), (unsigned)bz};
}

}  // namespace tsr950
