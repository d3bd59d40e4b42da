// Which products the few-row streaming kernels may read in place (host code, no device headers).
#pragma once
#include <algorithm>

namespace tsr950 {

// The 16-bit streaming kernel forms a lane's byte offsets inside a slice in 32 bits: a row of A from the
// slice's first column (read through a buffer range of 2^31 - 1 bytes, past which loads return zeros), and
// a row of the slice (32 rows of B) with the column, which would wrap at 2^32.  k itself stays an int, with a slice
// beyond the end of K still in range.  lda: A's own pitch, or that of the copy padded to a multiple of 8.
// 64 x 8 x 17,100,000 and 1 x 2^26 x 32 lie outside; such products take the paths that index in 64 bits.
inline bool few_rows16_in_range(int M, int N, int K, long lda, long ldb) {
  const long pitch_a = std::max(lda, ((long)K + 7) / 8 * 8);
  const long a_end = ((M - 1) * pitch_a + 8) * 2 + 32 + 16;            // lane half, second half of the slice, the load
  const long b_end = (31 * ldb + N) * 2;
  return K <= 0x7fffffff - 64 && a_end <= 0x7fffffffL && b_end <= 0xffffffffL;
}

}  // namespace tsr950
