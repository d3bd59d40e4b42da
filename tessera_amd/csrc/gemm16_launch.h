// Host-side tile selection and launch for the 16-bit MFMA GEMM family.
#pragma once
#include <algorithm>
#include <mutex>
#include "few_rows.h"
#include "gemm16.h"
#include "gemm16_skinny.h"
#include "host_util.h"
#include "pitch_copy.h"

namespace tsr950 {

// Any-shape fallback: one thread per output element, f32 accumulate in k order.
// Used when rows are not 16-byte aligned (K or N not a multiple of 8), where the
// vector loads of the MFMA kernel do not apply.
template <class T, int EPI>
__global__ void gemm16_generic_kernel(const Gemm16Params p) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  const int m = blockIdx.y * blockDim.y + threadIdx.y;
  const int z = blockIdx.z;
  if (m >= p.M || n >= p.N) return;
  const uint16_t* A = p.A + (long)z * p.strideA + (long)m * p.lda;
  const uint16_t* B = p.B + (long)z * p.strideB + n;
  float acc = 0.f;
  for (int k = 0; k < p.K; ++k) acc += from_storage<T>(A[k]) * from_storage<T>(B[(long)k * p.ldb]);
  if constexpr (EPI == EPI_GATED_F32) {
    const uint16_t* B2 = p.B2 + (long)z * p.strideB + n;
    float up = 0.f;
    for (int k = 0; k < p.K; ++k) up += from_storage<T>(A[k]) * from_storage<T>(B2[(long)k * p.ldb]);
    acc = activate(acc, p.act) * up;
  } else {
    if (p.bias) acc += p.bias[n];
    acc = activate(acc, p.act);
  }
  const long o = (long)z * p.strideD + (long)m * p.ldd + n;
  if constexpr (EPI == EPI_F32 || EPI == EPI_GATED_F32) reinterpret_cast<float*>(p.D)[o] = acc;
  else reinterpret_cast<uint16_t*>(p.D)[o] = to_storage<T>(acc);
}

// Grouped any-shape fallback: thread per output element, group found by scan.
template <class T, int EPI>
__global__ void gemm16_grouped_generic_kernel(const Gemm16Params p) {
  const int n = blockIdx.x * blockDim.x + threadIdx.x;
  const int m = blockIdx.y * blockDim.y + threadIdx.y;
  if (m >= p.M || n >= p.N) return;
  int e = 0;
  while (e + 1 < p.groups && m >= p.offsets[e + 1]) ++e;
  if (m < p.offsets[e] || m >= p.offsets[e + 1]) return;
  const uint16_t* A = p.A + (long)(p.gather ? p.gather[m] : m) * p.lda;
  const uint16_t* B = p.B + (long)e * p.strideB + n;
  float acc = 0.f;
  for (int k = 0; k < p.K; ++k) acc += from_storage<T>(A[k]) * from_storage<T>(B[(long)k * p.ldb]);
  if constexpr (EPI == EPI_SWIGLU16) {
    const uint16_t* B2 = p.B2 + (long)e * p.strideB + n;
    float up = 0.f;
    for (int k = 0; k < p.K; ++k) up += from_storage<T>(A[k]) * from_storage<T>(B2[(long)k * p.ldb]);
    const float gs = from_storage<T>(to_storage<T>(acc));
    const float us = from_storage<T>(to_storage<T>(up));
    acc = swiglu_of(gs, us);
  }
  const long o = (long)m * p.ldd + n;
  if constexpr (EPI == EPI_F32) reinterpret_cast<float*>(p.D)[o] = acc;
  else reinterpret_cast<uint16_t*>(p.D)[o] = to_storage<T>(acc);
}

// The 256 x 256 workgroup tiles, dense and grouped (per expert), use the 16-wide MFMA in the
// register-staged main loop; the smaller tiles use the 32-wide one.
constexpr int kBigTileMfma = 16;
constexpr int kGroupedTileMfma = 16;

inline bool aligned16(const void* p) { return (reinterpret_cast<uintptr_t>(p) & 15) == 0; }

// wg_limit > 0: only the first wg_limit workgroups of a dense product's tile order are launched
// (the caller serves the remaining tiles itself).
template <class T, int BM, int BN, int WM, int WN, int EPI, bool GROUPED, int MS = 32, bool MID = false, bool NTB = false>
int launch_gemm16_tile(Gemm16Params p, hipStream_t s, int wg_limit = 0) {
  constexpr int kLds = gemm16_paired_tail<BM, WM * WN, GROUPED, MID>() ? std::max(Gemm16Smem<BM, BN>::kBytes, Gemm16Smem<64, 2 * BN>::kBytes)
                                                                       : Gemm16Smem<BM, BN>::kBytes;
  auto kern = gemm16_kernel<T, BM, BN, WM, WN, EPI, GROUPED, MS, MID, NTB>;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(once, [&] {
    attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, kLds);
  });
  if (attr_err != hipSuccess) return kDeviceFailed;
  constexpr int BN_OUT = (EPI == EPI_SWIGLU16 || EPI == EPI_GATED_F32) ? BN / 2 : BN;
  p.tiles_n = ceil_div(p.N, BN_OUT);
  dim3 grid;
  if constexpr (GROUPED) {
    // every group contributes at most ceil(rows/BM) <= rows/BM + 1 tiles
    // (+8: the kernel deals ceil(real tiles / 8) slots to each of the 8 XCDs)
    p.tiles_m = p.M / BM + p.groups;
    grid = dim3(p.tiles_n * p.tiles_m + 8, 1, 1);
  } else {
    p.tiles_m = ceil_div(p.M, BM);
    grid = dim3(wg_limit > 0 ? wg_limit : p.tiles_m * p.tiles_n, 1, p.groups);
  }
  hipLaunchKernelGGL(kern, grid, dim3(WM * WN * 64), kLds, s, p);
  return launch_status();
}

// D[m][n] = sum over splits (in split order) of the f32 partials ws[splits][M][ldw], then bias and activation,
// stored as f32 or in the storage dtype; four columns per thread.
template <class T, int EPI>
__global__ void splitk_reduce_kernel(const float* __restrict__ ws, void* __restrict__ D, int M, int N, long ldw, long ldd,
                                     int splits, const float* __restrict__ bias, int act, int vec) {
  const long i = (long)blockIdx.x * blockDim.x + threadIdx.x;
  const int nq = (N + 3) / 4;
  if (i >= (long)M * nq) return;
  const int m = (int)(i / nq), n = (int)(i % nq) * 4;
  const size_t slice = (size_t)M * ldw;
  // (the partials of four splits are fetched together: they were written by other
  // XCDs, so every one of these loads pays a trip to memory)
  float4 acc = make_float4(0.f, 0.f, 0.f, 0.f);
  for (int z0 = 0; z0 < splits; z0 += 4) {
    float4 v[4];
#pragma unroll
    for (int u = 0; u < 4; ++u)
      v[u] = z0 + u < splits ? *reinterpret_cast<const float4*>(ws + (z0 + u) * slice + (size_t)m * ldw + n)
                             : make_float4(0.f, 0.f, 0.f, 0.f);
#pragma unroll
    for (int u = 0; u < 4; ++u) { acc.x += v[u].x; acc.y += v[u].y; acc.z += v[u].z; acc.w += v[u].w; }
  }
  store_quad<T, EPI>(D, (long)m * ldd, n, N, acc, bias, act, vec);
}
template <class T, int EPI>
int launch_splitk_reduce(const float* ws, long ldw, const Gemm16Params& p, int splits, int vec, hipStream_t s) {
  const long quads = (long)p.M * ((p.N + 3) / 4);
  hipLaunchKernelGGL((splitk_reduce_kernel<T, EPI>), dim3((unsigned)((quads + 255) / 256)), dim3(256), 0, s, ws, p.D, p.M,
                     p.N, ldw, p.ldd, splits, p.bias, p.act, vec);
  return launch_status();
}

// Tile and split-K choice of the dense 16-bit GEMM for an aligned problem — the one
// place the decision lives (the launcher below and the schedule query of the C ABI
// both call it).
struct Gemm16Schedule {
  int tile;      // workgroup tile edge: 256, 128 or 64 (square unless tile_m says otherwise)
  int split_k;   // number of K splits (1 = none)
  bool skinny;   // the few-row streaming kernel (32 x 64 workgroup tile up to 8 rows, 32 x 128 above; K slices of 32)
  int rest_split = 1;   // 256 tiles, split_k 1: K splits of the tiles beyond the last full round of 256
  int pieces = 1;       // ... or 2 or 4: pieces of the output these tiles are cut into
  int tile_m = 0;       // 128 with tile 256: the 128 x 256 tile (tile rows x tile columns); 0: square
};
constexpr int kSkinnyMaxM = 8;           // 64-column strips up to here,
constexpr int kSkinnyWideMaxM = 32;      // 128-column strips up to here
constexpr int kLooseMaxM = 64;           // and for rows of B on any boundary up to here
constexpr long kSplitTargetWgs = 768;
constexpr int kWeightStreamMaxM = 128;   // up to here a product is bound by reading B once

// K steps in each part of a K split: as many in every part but the last, which may be shorter.  (A split used to need a
// K that it divides into whole steps: 202 x 5120 x 9152 stayed whole, 93 us, and
// takes 42 in three; 961 x 960 x 11344 84 -> 37, 64 x 896 x 14000 82 -> 14.)
inline int split_steps(int K, int splits) { return ceil_div(ceil_div(K, G16_BK), splits); }
inline bool can_split(int K, int splits) { return (long)(splits - 1) * split_steps(K, splits) < ceil_div(K, G16_BK); }

// Time estimates (microseconds) behind the choice for products with more than kWeightStreamMaxM
// rows, fitted to timings of forced (tile, split) pairs on this part over products from 1024^3
// to 7168^3: a 256 x 256 tile spends 9.6 us outside its K loop and 1.09 us per 64-deep K step
// while at most 144 of the 256 compute units are busy, rising to 1.43 us with all of them busy
// (the board's power limit sets the clock); a 128 x 128 tile 5 us and 0.52 us per step, two
// of them sharing a compute unit at half that rate each (512 run at a time); the sum over K splits reads the f32
// partials and writes the result at about 4.4 TB/s.
inline double est_tiles256_us(long tiles, int ksteps) {
  const long full = tiles / 256, rem = tiles % 256;
  double t = (double)full * (9.6 + ksteps * 1.43);
  if (rem) t += 9.6 + ksteps * (1.09 + 0.34 * std::min(1.0, std::max(0.0, (rem - 144) / 112.0)));
  return t;
}
// (a 128 x 256 tile: 7 us and 0.60 us per step up to about 96 tiles at a time, 0.82 with every
// compute unit busy over several rounds — per FLOP a fifth slower than the 256 x 256 tile, but
// twice as many tiles to fill the chip with; a single partial round of 160 to 255 tiles measured
// 0.83 to 0.93 per step)
inline double est_tiles128x256_us(long tiles, int ksteps) {
  const long full = tiles / 256, rem = tiles % 256;
  double t = (double)full * (7.0 + ksteps * 0.82);
  if (rem) t += 7.0 + ksteps * (0.60 + 0.28 * std::min(1.0, std::max(0.0, (rem - 96) / 64.0)));
  return t;
}
inline double est_tiles128_us(long tiles, int ksteps) {
  return 5.0 * (double)((tiles + 511) / 512) + ksteps * 0.52 * (double)((tiles + 255) / 256);
}
inline double est_split_sum_us(long mn, int splits) {
  return splits > 1 ? 2.0 + (double)mn * (4.0 * splits + 2.0) / 4.4e6 : 0.0;
}

// Time estimate (microseconds) for 33 to 128 rows against a weight matrix that streams from HBM,
// fitted (13 % rms) to timings of forced (tile, split) pairs on this part over 19 weight shapes from
// 2048 x 7168 to 32768 x 4096 with the weights cycled through copies: a launch cost, then the larger
// of the busiest compute unit's K steps (its first workgroup at `step`, every further one sharing
// the unit at `shared` per step) and the time to stream the tile columns of B at `tbs` TB/s, which
// takes about 185 workgroups in flight to reach; a split adds 3.4 us and 1.6 us per million
// partial sums.
struct FewRowTile { int tile_m, tile_n; double launch, step, shared, tbs; };
constexpr FewRowTile kFewRowTiles[3] = {{64, 64, 0.26, 0.514, 0.256, 5.39},
                                        {128, 128, 2.31, 0.345, 0.728, 5.46},
                                        {128, 256, 3.97, 0.693, 1.582, 7.01}};
inline double est_few_rows_us(const FewRowTile& t, int M, int N, int K, int splits) {
  const long wgs = (long)ceil_div(M, t.tile_m) * ceil_div(N, t.tile_n) * splits;
  const double steps = split_steps(K, splits);
  const double busiest = (double)((wgs + 255) / 256);
  const double compute = steps * (t.step + t.shared * (busiest - 1.0));
  const double bytes = 2.0 * K * ceil_div(N, t.tile_n) * t.tile_n;
  const double stream = bytes / (t.tbs * 1e6 * std::min(1.0, wgs / 185.0));
  const double sum = splits > 1 ? 3.4 + (double)M * N * splits * 1.6e-6 : 0.0;
  return t.launch + std::max(compute, stream) + sum;
}

// Second opinion for single products of more than 128 rows on fewer than 260 tiles of 256 x 256, where the estimates
// above (fitted to matrices found in the caches, in equal K parts, and without the 64 x 64 tile) were on average 5.6 % behind the
// best of the forced schedules and up to 47 %: fitted (4 to 12 % rms) to 2033 timings of forced (tile, split) pairs over 260
// products of 129 to 3000 rows, weights streamed from memory.  A launch, then the larger of the K steps and of streaming B;
// 64- and 128-wide tiles share a compute unit (the first at `step` a K step, each further one `more`), 256-wide ones come in
// rounds (a step `step` on a quiet chip, `more` on a full one); a split adds its sum.  (The figures are a fit and not rates of the
// part: 64-wide tiles hardly ever wait for B, hence their 14 TB/s.)
struct MidTile { int tile_m, tile_n; double launch, step, more, tbs, sum, per_mega; };
constexpr MidTile kMidTiles[4] = {{64, 64, 1.158, 0.4031, 0.1924, 14.09, 2.744, 1.677},
                                  {128, 128, 2.436, 0.5124, 0.5325, 2.914, 3.348, 1.262},
                                  {128, 256, 3.896, 0.749, 1.006, 5.977, 3.825, 0.9554},
                                  {256, 256, 8.098, 1.089, 1.506, 6.356, 4.376, 0.8394}};
inline double est_mid_us(const MidTile& t, int M, int N, int K, int splits) {
  const long wgs = (long)ceil_div(M, t.tile_m) * ceil_div(N, t.tile_n) * splits;
  const double per = split_steps(K, splits);
  const double bytes = 2.0 * K * ceil_div(N, t.tile_n) * t.tile_n;
  const double stream = t.launch + bytes / (t.tbs * 1e6 * std::min(1.0, wgs / 185.0));
  double steps;
  if (t.tile_n < 256) {
    steps = t.launch + per * (t.step + t.more * (double)((wgs + 255) / 256 - 1));
  } else {
    const double rest = (double)(wgs % 256);
    steps = (double)(wgs / 256) * (t.launch + per * t.more);
    if (rest > 0) steps += t.launch + per * (t.step + (t.more - t.step) * std::min(1.0, std::max(0.0, (rest - 96.0) / 128.0)));
  }
  return std::max(steps, stream) + (splits > 1 ? t.sum + (double)M * N * splits * t.per_mega * 1e-6 : 0.0);
}
// The schedule `first` or, where this estimate sees a tenth less time, its own choice.  `equal` is what the first estimate chose
// without K parts of unequal length, to which it was not fitted: where `first` has such parts, they are dropped unless this one, too,
// sees them ahead (1228 x 1112 x 1472 whole 27.8 us, in three parts 33.6; 255 x 3648 x 9792 in four unequal parts 37.9, in three equal
// ones 43.6; not for the best whole tile instead, whatever the parts: 754 x 4376 x 11136 went from 96 us in three equal parts to 126 so, and takes
// 91 in four).  4800 drawn products of 129 rows and more, each timed under all its schedules: where this check changes the choice, 124
// times, 6 % faster on average, 23 of them more than 3 % slower.  (Asked for a microsecond's gain: 130, 5 %, 30.)
// Above 3000 rows, which it was not fitted to either, it is asked for unequal parts alone, and 5 % are enough, as the first
// estimate is the more careful one with those (6782 x 768 x 13040 215 us whole, 135 in three parts).
inline Gemm16Schedule second_opinion_mid(const Gemm16Schedule& first, const Gemm16Schedule& equal, int M, int N, int K) {
  auto is = [](const MidTile& t, const Gemm16Schedule& s) { return t.tile_n == s.tile && t.tile_m == (s.tile_m ? s.tile_m : s.tile); };
  auto unequal = [K](int splits) { return splits > 1 && K % (splits * G16_BK) != 0; };
  const bool fitted = M <= 3000;
  double first_us = 0.0, equal_us = 0.0, best_us = 1e30;
  Gemm16Schedule best = first;
  for (const MidTile& t : kMidTiles) {
    if (is(t, first)) first_us = est_mid_us(t, M, N, K, first.split_k);
    if (is(t, equal)) equal_us = est_mid_us(t, M, N, K, equal.split_k);
    if (t.tile_n == 64 && M > 512) continue;           // (not measured)
    for (int splits : {1, 2, 3, 4, 6, 8}) {
      if (splits > 1 && (!can_split(K, splits) || K / splits < 256)) continue;
      if (!fitted && !unequal(splits)) continue;
      const double us = est_mid_us(t, M, N, K, splits);
      if (us < best_us) {
        best_us = us;
        best = t.tile_m < t.tile_n ? Gemm16Schedule{256, splits, false, 1, 1, 128} : Gemm16Schedule{t.tile_n, splits, false};
      }
    }
  }
  // (from a 256-wide tile to 128 x 128 ones, whose third and fourth on a unit cost more than the estimate has them, by a
  // fifth; to more parts by 2 us at least: 1052 x 704 x 1472 in four parts 14.9 us, whole 12.5)
  const double margin = first.tile == 256 && best.tile < 256 ? 0.8 : fitted ? 0.9 : 0.95;
  if (best_us < margin * first_us && (best.split_k <= first.split_k || best_us + 2.0 < first_us)) return best;
  return fitted && unequal(first.split_k) && equal_us < first_us ? equal : first;
}

// Stacks of products whose 128 x 128 tiles leave half of the compute units idle go on 64 x 64 ones, while K is short: a
// step of those reads twice the operands per result, from the caches all of them share.  (90 stacks of 2 to 64 products of
// 16 to 1024 rows, forced: on average 2 % behind the best tile instead of 12, none more than 4 % behind what it had; 4 of
// 124 x 560 x 176 5.0 -> 3.4 us, 4 of 128 x 256 x 64 4.2 -> 3.4, on the device; a caller in Python sees 4.2 either way, the call's host path.  13 of 141 x 376 x 704 9.3 us on 128 x 128, 10.0 on 64 x 64; 25 of 384 x 256 x 448, 150 tiles, 8.8 and 10.9.)
inline bool small_tiles_for_stack(long tiles128, int K, int batch) { return batch > 1 && tiles128 < 128 && K <= 640; }

// Workgroups of the few-row kernel on 128-column strips with K in as many parts as keep it within one workgroup
// per compute unit (a second round would be nearly empty), every wave with at least one slice.
inline int skinny_wide_splits(int N, int K) {
  return std::max(1, std::min(256 / ceil_div(N, 128), K / 256));
}
// K splits for rows of B on any boundary, where the streaming kernel is the only one that reads B in place:
// the fewest microseconds by an estimate fitted to forced splits over 512 to 16384 columns and 256 to
// 14336 rows of B (a workgroup streams a 256-byte row in 7.5 ns, the chip 5.6 TB/s; a split adds a launch
// and a sum, 3.6 us).
inline int skinny_loose_splits(int N, int K) {
  const int strips = ceil_div(N, 128), most = skinny_wide_splits(N, K);
  int best = 1;
  double best_us = 1e30;
  for (int splits = 1; splits <= most; ++splits) {
    const double rounds = ceil_div(strips * splits, 256) * 256.0 / std::max(256, strips * splits);
    const double us = std::max(7.5e-3 * K / splits, 2.0 * K * N / 5.6e6) * rounds + (splits > 1 ? 3.6 : 0.0);
    if (us < best_us) { best_us = us; best = splits; }
  }
  return best;
}

// A few rows (a B that streams from memory), K in `splits` parts of unequal length or in the `equal` ones that divide it.  Equal
// ones where they are at least two thirds as many (21 x 10272 x 2816 in five / four parts 20.0 / 18.5 us), and short ones
// that are 360 workgroups by themselves (27 x 10240 x 3264 in five / three 17.5 / 15.8; 16 x 8320 x 5952, three of 1984,
// 22.2 / 27.0).  Whole instead of two parts that save less than their sum costs: 18 x 2176 x 1088 whole / in two 6.4 / 8.2, 12 x 640 x
// 1344 7.2 / 8.6, 9 x 1728 x 1472 9.3 / 7.6; sooner over many columns, where a second workgroup on each unit streams B
// faster (2 x 2952 x 1384 1.16 times as fast in two), and over more than 1100 off 128-byte lines (49 x 1128 x 1472 10.2 / 8.8, 17 x
// 2120 x 1176 8.9 / 8.3).  Where 64-wide tiles fill the chip by themselves the lines count the other way (31 x
// 13072 x 1368 13.3 / 14.1, 13 x 14704 x 1648 15.0, in three 16.8; 14 x 13504 x 1984 16.2, in three 13.6).
// Under 128 columns (router logits) always in parts: in a layer such a product's operands come from memory (762 x 32 x 1344 in front
// of its experts 14 us whole, 11 in two parts; 2000 times the same one 7.3 and 8.6).
// Drawn products of up to 64 rows, libraries with and without unequal parts in turn: with them 1.20 times as fast, 12 of 827 more than 3 %
// slower.
// (These lines stand between times of calls repeated on one matrix, from the caches, where the second launch counts in full.  With weights
// from memory and the launches queued up two parts are ahead below them too, 7 % on average over 41 drawn products, 18 x 2176 x
// 1088 and its like by 0.5 us; with weights from memory called one by one, level over 43.)
inline bool unequal_parts_pay(long tiles, int N, int K, int splits, int equal) {
  const bool lines = N % 64 == 0;
  if (3 * equal >= 2 * splits) return false;
  if (N < 128) return true;
  if (equal > 1) return tiles * equal < 360 || K / equal >= 1536;
  if (tiles >= 200) return K >= (lines ? 1200 : 2048);
  return splits > 2 || K >= (!lines && tiles >= 18 ? 1160 : tiles < 24 ? 1480 : tiles < 40 ? 1400 : 1088);
}

inline Gemm16Schedule select_gemm16_schedule(int M, int N, int K, int batch) {
  if (batch == 1 && M <= kWeightStreamMaxM && N >= 128) {
    // Few rows under a very wide weight matrix (a vocabulary projection, a fused up projection):
    // tiles enough for three quarters of the compute units without a K split, which would add a
    // pass over the partials and little parallelism.  The wider tile reads 512 contiguous bytes
    // of a row of B instead of 256 and streams faster once it, too, fills the chip.
    if ((long)ceil_div(M, 128) * ceil_div(N, 256) >= 192) return {256, 1, false, 1, 1, 128};
    if ((long)ceil_div(M, 128) * ceil_div(N, 128) >= 192) return {128, 1, false};
  }
  if (batch == 1 && M <= kSkinnyMaxM && K % 32 == 0 && K >= 512) {
    // one workgroup per 64-column strip and K split; about one workgroup per CU, and
    // at least two 32-row slices for each of a workgroup's 8 waves
    const int strips = ceil_div(N, 64);
    int splits = std::max(1, std::min((256 + strips / 2) / strips, K / 512));
    return {64, splits, true};
  }
  if (batch == 1 && M > 32 && M <= kWeightStreamMaxM && N >= 2048 && K >= 1024) {
    // the cheapest of the three small tiles with K in 1 to 16 parts, by the estimate above (below
    // 33 rows the rule further down is as good as the estimate: 1 % apart over the same shapes)
    Gemm16Schedule best{128, 1, false};
    double best_us = 1e30;
    for (const FewRowTile& t : kFewRowTiles)
      for (int splits : {1, 2, 3, 4, 6, 8, 12, 16}) {
        if (!can_split(K, splits) || K / splits < 512) continue;
        // (the estimate was fitted to equal parts; others have to be worth a twelfth: 84 x 4864 x 1600 whole / in three
        // parts 11.3 / 12.6 us)
        const double us = est_few_rows_us(t, M, N, K, splits) * (K % (splits * G16_BK) != 0 && splits > 1 ? 1.08 : 1.0);
        if (us < best_us) {
          best_us = us;
          best = t.tile_n == 256 ? Gemm16Schedule{256, splits, false, 1, 1, 128} : Gemm16Schedule{t.tile_m, splits, false};
        }
      }
    return best;
  }
  const long tiles256 = (long)ceil_div(M, 256) * ceil_div(N, 256) * batch;
  const long tiles128 = (long)ceil_div(M, 128) * ceil_div(N, 128) * batch;
  if (M > kWeightStreamMaxM && N >= 128) {
    // the cheapest of: either tile, K in 1, 2, 3, 4 or 8 parts of at least 512 (a single product only)
    const int ksteps = ceil_div(K, G16_BK);
    Gemm16Schedule best{256, 1, false};
    double best_us = est_tiles256_us(tiles256, ksteps);
    auto consider = [&](int tile, int splits, double us) {
      if (us < best_us) { best_us = us; best = Gemm16Schedule{tile, splits, false}; }
    };
    consider(128, 1, est_tiles128_us(tiles128, ksteps));
    {
      // (its estimate is the least certain of the three — the per-step figure moved by 13 % between
      // shapes of equal tile count — so it has to win by a margin)
      const double us = 1.06 * est_tiles128x256_us((long)ceil_div(M, 128) * ceil_div(N, 256) * batch, ksteps);
      if (us < best_us) { best_us = us; best = Gemm16Schedule{256, 1, false, 1, 1, 128}; }
    }
    Gemm16Schedule equal = best, uneven = best;
    if (batch == 1) {
      double uneven_us = 1e30;
      for (int splits : {2, 3, 4, 8}) {
        const bool in_equal_parts = K % (splits * G16_BK) == 0;
        if (!can_split(K, splits) || K / splits < (in_equal_parts || M <= 3000 ? 512 : 1024)) continue;
        const double sum_us = est_split_sum_us((long)M * N, splits);
        const double us256 = est_tiles256_us(tiles256 * splits, split_steps(K, splits)) + sum_us;
        const double us128 = est_tiles128_us(tiles128 * splits, split_steps(K, splits)) + sum_us;
        if (in_equal_parts) {
          consider(256, splits, us256);
          consider(128, splits, us128);
        } else {
          if (us256 < uneven_us) { uneven_us = us256; uneven = {256, splits, false}; }
          if (us128 < uneven_us) { uneven_us = us128; uneven = {128, splits, false}; }
        }
      }
      // The estimates were fitted without parts of unequal length.  Up to 3000 rows the second opinion below looks at these again;
      // above, parts are at least 1024 deep (3077 x 640 x 1848 whole / in two parts 17.5 / 21.9 us) and have to win by half a
      // microsecond, by 4 % against equal ones, and by 14 % against whole 128 x 256 tiles, whose estimate is 10 to 25 %
      // high while they are one round of the chip (3170 x 1728 x 3520 whole / in two parts 46 / 56 us).  Over 380 products of
      // more than 3000 rows, timed as those of the second opinion: 0.6 % behind on average, 15 % at most.
      equal = best;
      const bool take = M <= 3000 ? uneven_us < best_us
                                  : (best.tile_m ? 1.14 : best.split_k > 1 ? 1.04 : 1.0) * uneven_us + 0.5 < best_us;
      if (take) { best_us = uneven_us; best = uneven; }
    }
    // A tile count that is not a multiple of 256 leaves compute units idle in the last round: its tiles can be cut into
    // two or four pieces, or, where they are few and K is long, split along K among those units (one more launch and
    // a sum over the partial tiles: 16 tiles left at K = 4096 137 against 139 us in pieces, at K = 14336 406 against 489;
    // 80 left at K = 4096 185 against 177).  Pieces still have a whole round before them: under 12 K steps, where prologue and
    // epilogue are most of it, they have to win against 128 x 128 tiles, two on a unit, by a fifth (5860 x 3424 x 520 with
    // gelu 51 us on those, 58 in pieces).
    const long full = tiles256 / 256, rest = tiles256 % 256;
    if (batch == 1 && full >= 1 && rest > 0 && rest <= 128 && tiles256 < (1L << 30)) {
      const double main_us = (double)full * (9.6 + ksteps * 1.43);
      const double margin = best.tile == 128 && ksteps < 12 ? 1.2 : 1.0;
      auto cut = [&](int pieces, double us) {
        us *= margin;
        if (us < best_us) { best_us = us; best = Gemm16Schedule{256, 1, false, 1, pieces}; }
      };
      // (128 x 256 pieces beside whole tiles: no less than 0.72 us a K step, on idle compute units too: 49 tiles left at K = 4832 in
      // two / four pieces or four K parts 196 / 192 / 185 us; 0.60 sent 7521 x 2368 x 4824 from 172 us in K parts to 195 in two pieces)
      cut(2, main_us + std::max(est_tiles128x256_us(2 * rest, ksteps), 7.0 + 0.72 * ksteps));
      // (128 x 128 pieces, alone on their compute units: 0.52 us a K step up to 64 of them, 0.65 from 192 on)
      if (rest <= 64) cut(4, main_us + 5.0 + ksteps * (0.52 + 0.13 * std::min(1.0, std::max(0.0, (4 * rest - 64) / 128.0))));
      for (int splits : {2, 3, 4, 6, 8, 12, 16}) {
        const int per = ceil_div(ksteps, splits);
        if (rest * splits > 256 || per < 2 || (long)per * (splits - 1) >= ksteps) continue;
        // (the partials of a few tiles are summed from the caches)
        const double us = main_us + 8.0 + est_tiles256_us(rest * splits, per) + 0.9 * est_split_sum_us(rest * 65536L, splits);
        if (us < best_us) { best_us = us; best = Gemm16Schedule{256, 1, false, splits}; }
      }
    }
    if (batch == 1 && tiles256 < 260 && best.rest_split == 1 && best.pieces == 1)
      best = second_opinion_mid(best, equal, M, N, K);
    if (best.tile <= 128 && small_tiles_for_stack(tiles128, K, batch)) best.tile = 64;
    return best;
  }
  // Few rows: the weight matrix streams from HBM once and the tiles are small; for a single
  // product with few tiles and a long K, K is split over about 768 workgroups.
  if (tiles256 >= 192) return {256, 1, false};
  if (batch == 1 && M > 64 && M <= kWeightStreamMaxM && N >= 128 && N < 2048 && K <= 4608) {
    // 65 to 128 rows over few columns: 64 x 64 tiles, K in as many parts as the estimate of the mid sizes likes.  (Forced
    // schedules of 32 such products: on 128 x 128 tiles, the rule below, 23 % behind the best; 104 x 864 x 2376 14.0 -> 8.7
    // us, 100 x 2008 x 2176 13.5 -> 9.6.  From K = 4700 on the larger tile is level or ahead.)
    Gemm16Schedule best{64, 1, false};
    double best_us = 1e30;
    for (int splits : {1, 2, 3, 4, 6, 8}) {
      if (splits > 1 && (!can_split(K, splits) || K / splits < 256)) continue;
      const double us = est_mid_us(kMidTiles[0], M, N, K, splits);
      if (us < best_us) { best_us = us; best.split_k = splits; }
    }
    return best;
  }
  const bool t128 = tiles128 >= 192 || (M > 64 && N >= 128);
  int splits = 1;
  if (batch == 1) {
    const long tiles = t128 ? tiles128 : (long)ceil_div(M, 64) * ceil_div(N, 64);
    splits = (int)std::max<long>(1, std::min<long>((kSplitTargetWgs + tiles - 1) / tiles, K / 512));
    // the f32 partials are written and read once per split (8 M N splits bytes against
    // 2 K (M + N) bytes of operands: B dominates under few rows, A over few columns): beyond two
    // splits keep that under about 0.4 of the operand traffic
    splits = (int)std::min<long>(splits, std::max<long>(2, (long)K * (M + N) / (10L * M * N)));
    while (splits > 1 && !can_split(K, splits)) --splits;
    int equal = splits;
    while (equal > 1 && K % (equal * G16_BK) != 0) --equal;
    if (splits > equal && !unequal_parts_pay(tiles, N, K, splits, equal)) splits = equal;
    // 9 to 32 rows: the streaming kernel on 128-column strips instead where it streams faster than the tiles: one
    // workgroup on every compute unit (16 x 8192 x 8192 31.4 -> 28.1 us, 4096 x 4096 12.7 -> 11.3, 8192 x 2048 10.4 ->
    // 9.4; two parts of a short K, 16320 x 2560, 18.2 against 17.3), or nearly so and a B that is read with the
    // non-temporal hint (7168 x 8192 29.4 -> 25.7, 14336 x 4096 28.5 -> 25.6).  Else the tiles: 7168 x 4096 15.4 against
    // 13.0, 8064 x 4096 (252 workgroups) 16.2 against 14.1, 6144 x 8192 23.0 against 21.2, 14656 x 2176 15.4 against 13.9; with K ranges
    // under 512, 2048 x 7168, 11.5 against 12.2.  And where the parts of K leave the tiles
    // too few workgroups (9 x 3520 x 5312).  (The lines lie between those points, all but the last at 16 rows; 1.1e8 stands
    // above kStreamOnceBytes because 6144 x 8192, 1.007e8, gains nothing.  Over 16 weight shapes under 9 to 32 rows, several
    // matrices in turn, no choice is slower than the tiles by more than 1 %; a matrix alone in a loop: see kStreamOnceBytes.)
    // (Under 16 rows against the tiles' equal parts only: in unequal ones they lose there, 7 x 1280 x 2584 on strips 7.1 us, on tiles in five
    // parts 8.3, and win above, 19 x 896 x 9280 13.2 and 10.9.  A large B, too, stays with the strips where its rows are off 128-byte
    // lines, of which a 64-wide tile then reads one too many for every row, 30 x 6488 x 5384 21.0 us against 25.2, and from 9e7
    // bytes on, 25 x 6720 x 10904 30.9 and 34.5, 17 x 4480 x 11680 23.0 and 24.9; on the lines tiles win, in parts for about two workgroups
    // a unit, 20 x 3712 x 9528 17.9 and 15.5.)
    if (M <= kSkinnyWideMaxM && N >= 128) {
      const int wide = skinny_wide_splits(N, K);
      const long wgs = (long)ceil_div(N, 128) * wide;
      const double bytes = 2.0 * K * N;
      const bool streams = bytes >= 1.1e8 ? wgs >= 216 : bytes >= 2.4e7 && wgs >= 256 && wide > 2;
      auto strips = [&](int parts) {
        return (streams && wgs <= 256 && K >= 2048 && K / wide >= 512) || (K >= 2048 && tiles * parts < 128 && wgs > 2 * tiles * parts);
      };
      const bool equal_only = M < 16 || bytes >= 9e7 || (bytes >= 4.2e7 && N % 64 != 0);
      if (strips(equal_only ? equal : splits)) return {128, wide, true};
      if (splits > equal && strips(equal)) splits = std::max(equal, (int)std::min<long>(splits, 512 / tiles));
    }
  }
  return {t128 && !small_tiles_for_stack(tiles128, K, batch) ? 128 : 64, splits, false};
}

template <class T, int MI, int NW, int NJ, int EPI, bool NT, bool LOOSE>
int launch_gemm16_skinny_as(const Gemm16Params& p, int kps, int splits, float* part, int d_vec, hipStream_t s) {
  auto kern = gemm16_skinny_kernel<T, MI, NW, NJ, EPI, NT, LOOSE>;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(once, [&] {
    attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize,
                                   skinny_lds_bytes<NW, NJ>(32));
  });
  if (attr_err != hipSuccess) return kDeviceFailed;
  hipLaunchKernelGGL(kern, dim3(ceil_div(p.N, 32 * NJ), splits), dim3(NW * 64), (skinny_lds_bytes<NW, NJ>(std::min(p.M, 32))), s, p,
                     kps, part, d_vec);
  return launch_status();
}

// The few-row streaming kernel with K in `splits` parts.  loose: see the kernel; A is then copied into
// rows padded with zeros to a multiple of 8 where its own cannot be read 16 bytes at a time.  Without a
// workspace that is large enough (a capture on a stream with none or a smaller one) K stays whole; a copy of A without room is kNoScratch.
template <class T, int EPI>
int launch_gemm16_skinny(Gemm16Params p, int splits, bool loose, hipStream_t s) {
  const int cols = p.M <= kSkinnyMaxM && !loose ? 64 : 128;
  int kps = ceil_div(ceil_div(p.K, splits), 32) * 32;
  splits = ceil_div(p.K, kps);
  const long ldw = (long)ceil_div(p.N, cols) * cols;
  const int K8 = (p.K + 7) & ~7;
  const bool a_copy = loose && (p.K % 8 != 0 || p.lda % 8 != 0 || !aligned16(p.A));
  const size_t a_bytes = a_copy ? (((size_t)p.M * K8 * 2 + 255) & ~size_t(255)) : 0;
  const size_t part_bytes = splits > 1 ? (size_t)splits * p.M * ldw * 4 : 0;
  char* ws = nullptr;
  if (a_bytes + part_bytes) {
    ws = static_cast<char*>(stream_workspace_or_null(s, a_bytes + part_bytes));
    if (!ws && a_copy) return kNoScratch;
    if (!ws) { splits = 1; kps = ceil_div(p.K, 32) * 32; }
  }
  float* part = splits > 1 ? reinterpret_cast<float*>(ws + a_bytes) : nullptr;
  constexpr int dsz = EPI == EPI_F32 ? 4 : 2;
  const int d_vec = p.N % 4 == 0 && (p.ldd * dsz) % (4 * dsz) == 0 && aligned16(p.D) && (!p.bias || aligned16(p.bias));
  Gemm16Params q = p;
  if (a_copy) {
    PadLaunch<uint16_t> pad(1);
    pad.add({reinterpret_cast<uint16_t*>(ws), K8, 0, p.A, p.lda, 0, p.M, p.K, p.M});
    pad.run(s);
    if (int rc = launch_status(); rc != kOk) return rc;
    q.A = reinterpret_cast<const uint16_t*>(ws);
    q.lda = K8;
  }
  const bool nt = 2.0 * p.K * p.N >= kStreamOnceBytes;
  int rc;
  // (loose: off the 128-byte grid a row's piece lies in two cache lines and neighbouring strips want the same line, and
  // eight waves with a workgroup's whole K range in flight read at half the rate.  16 rows, eight / four waves / copies
  // into aligned buffers: N 8191 x K 4097 64 / 35 / 67 us, 14335 x 2049 56 / 30 / 49, 12001 x 12003 149 / 99 / 253)
  if (loose)
    rc = p.M <= 32 ? launch_gemm16_skinny_as<T, 1, 4, 4, EPI, false, true>(q, kps, splits, part, d_vec, s)
                   : launch_gemm16_skinny_as<T, 2, 4, 4, EPI, false, true>(q, kps, splits, part, d_vec, s);
  else if (cols == 64)
    rc = nt ? launch_gemm16_skinny_as<T, 1, 8, 2, EPI, true, false>(q, kps, splits, part, d_vec, s)
            : launch_gemm16_skinny_as<T, 1, 8, 2, EPI, false, false>(q, kps, splits, part, d_vec, s);
  else
    rc = nt ? launch_gemm16_skinny_as<T, 1, 8, 4, EPI, true, false>(q, kps, splits, part, d_vec, s)
            : launch_gemm16_skinny_as<T, 1, 8, 4, EPI, false, false>(q, kps, splits, part, d_vec, s);
  if (rc != kOk || !part) return rc;
  return launch_splitk_reduce<T, EPI>(part, ldw, p, splits, d_vec, s);
}

template <class T, int EPI>
int launch_gemm16(Gemm16Params p, hipStream_t s);

// A product whose operands the tile kernels cannot load as they are (K, N or a pitch not a
// multiple of 8 elements, or a pointer off a 16-byte boundary): the offending operands are
// copied into aligned, zero-padded buffers (K and N rounded up to multiples of 8: zero columns
// of A, zero rows and columns of B), the tile kernels run on those, and the leading N columns
// of the result are copied out.  The buffers live from here to the end of this call's work on
// the stream (stream-ordered allocation).
template <class T, int EPI>
int launch_gemm16_repitched(const Gemm16Params& p, hipStream_t s) {
  constexpr int dsz = (EPI == EPI_F32) ? 4 : 2;
  const int K8 = (p.K + 7) & ~7, N8 = (p.N + 7) & ~7, G = p.groups;
  const bool a_ok = p.K % 8 == 0 && p.lda % 8 == 0 && p.strideA % 8 == 0 && aligned16(p.A) && p.lda < (1L << 21);
  const bool b_ok = p.K % 8 == 0 && p.N % 8 == 0 && p.ldb % 8 == 0 && p.strideB % 8 == 0 && aligned16(p.B) &&
                    p.ldb < (1L << 21);
  const bool d_ok = p.N % 8 == 0 && (p.ldd * dsz) % 16 == 0 && (p.strideD * dsz) % 16 == 0 && aligned16(p.D);
  const bool bias_ok = !p.bias || (p.N % 8 == 0 && aligned16(p.bias));
  const size_t a_bytes = a_ok ? 0 : (size_t)G * p.M * K8 * 2, b_bytes = b_ok ? 0 : (size_t)G * K8 * N8 * 2;
  const size_t d_bytes = d_ok ? 0 : (size_t)G * p.M * N8 * dsz, bias_bytes = bias_ok ? 0 : (size_t)N8 * 4;
  char* ws = nullptr;
  if (!device_malloc_async(reinterpret_cast<void**>(&ws), a_bytes + b_bytes + d_bytes + bias_bytes + 16, s)) return kDeviceFailed;
  Gemm16Params q = p;
  q.K = K8;
  q.N = N8;
  PadLaunch<uint16_t> pad(G);
  char* at = ws;
  if (!a_ok) {
    uint16_t* a2 = reinterpret_cast<uint16_t*>(at);
    at += a_bytes;
    pad.add({a2, K8, (long)p.M * K8, p.A, p.lda, p.strideA, p.M, p.K, p.M});
    q.A = a2; q.lda = K8; q.strideA = (long)p.M * K8;
  }
  if (!b_ok) {
    uint16_t* b2 = reinterpret_cast<uint16_t*>(at);
    at += b_bytes;
    pad.add({b2, N8, (long)K8 * N8, p.B, p.ldb, p.strideB, p.K, p.N, K8});
    q.B = b2; q.ldb = N8; q.strideB = (long)K8 * N8;
  }
  void* d2 = nullptr;
  if (!d_ok) {
    d2 = at;
    at += d_bytes;
    q.D = d2; q.ldd = N8; q.strideD = (long)p.M * N8;
  }
  if (!bias_ok) {
    float* bias2 = reinterpret_cast<float*>(at);
    pad.add_vector(bias2, N8, p.bias, p.N);
    q.bias = bias2;
  }
  pad.run(s);
  int rc = launch_status();
  if (rc == kOk) rc = launch_gemm16<T, EPI>(q, s);
  if (rc == kOk && !d_ok) {
    if constexpr (dsz == 4)
      hipLaunchKernelGGL(unpad_rows_kernel<float>, copy_grid(p.M, N8, 4, G), copy_block(), 0, s, static_cast<float*>(p.D),
                         p.ldd, p.strideD, static_cast<const float*>(d2), (long)N8, (long)p.M * N8, p.M, p.N);
    else
      hipLaunchKernelGGL(unpad_rows_kernel<uint16_t>, copy_grid(p.M, N8, 8, G), copy_block(), 0, s,
                         static_cast<uint16_t*>(p.D), p.ldd, p.strideD, static_cast<const uint16_t*>(d2), (long)N8,
                         (long)p.M * N8, p.M, p.N);
    rc = launch_status();
  }
  if (hipFreeAsync(ws, s) != hipSuccess) { (void)hipGetLastError(); rc = rc == kOk ? kDeviceFailed : rc; }
  return rc;
}

// The tiles first_tile .. first_tile + rest - 1 of a dense product on 256 x 256 tiles, each split
// along K over `splits` workgroups into ws, then summed (with the bias / activation of the product).
template <class T, int EPI>
int launch_gemm16_rest(Gemm16Params p, int first_tile, int rest, int splits, float* ws, hipStream_t s) {
  using S = Gemm16Smem<256, 256>;
  auto kern = gemm16_rest_splitk_kernel<T, kBigTileMfma>;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(once, [&] {
    attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern),
                                   hipFuncAttributeMaxDynamicSharedMemorySize, S::kBytes);
  });
  if (attr_err != hipSuccess) return kDeviceFailed;
  p.tiles_m = ceil_div(p.M, 256);
  p.tiles_n = ceil_div(p.N, 256);
  const int ksplit = ceil_div(ceil_div(p.K, G16_BK), splits) * G16_BK;
  hipLaunchKernelGGL(kern, dim3(rest, splits), dim3(256), S::kBytes, s, p, first_tile, ksplit, ws);
  if (int rc = launch_status(); rc != kOk) return rc;
  hipLaunchKernelGGL((gemm16_rest_sum_kernel<T, EPI>), dim3(64, rest), dim3(256), 0, s, ws, p.D, p.M, p.N, p.ldd,
                     p.tiles_m, p.tiles_n, first_tile, splits, p.bias, p.act);
  return launch_status();
}

// A dense product on 256 x 256 tiles with those beyond the last full round of 256 in `pieces` pieces each.
template <class T, int EPI>
int launch_gemm16_pieces(Gemm16Params p, int pieces, hipStream_t s) {
  using S = Gemm16Smem<256, 256>;
  auto kern = gemm16_pieces_kernel<T, EPI>;
  static std::once_flag once;
  static hipError_t attr_err = hipSuccess;
  std::call_once(once, [&] {
    attr_err = hipFuncSetAttribute(reinterpret_cast<const void*>(kern), hipFuncAttributeMaxDynamicSharedMemorySize, S::kBytes);
  });
  if (attr_err != hipSuccess) return kDeviceFailed;
  p.tiles_m = ceil_div(p.M, 256);
  p.tiles_n = ceil_div(p.N, 256);
  const int tiles = p.tiles_m * p.tiles_n, main_tiles = tiles / 256 * 256, rest = tiles - main_tiles;
  hipLaunchKernelGGL(kern, dim3(main_tiles + ceil_div(rest, 8) * 8 * pieces), dim3(256), S::kBytes, s, p, main_tiles, pieces);
  return launch_status();
}

// Dense / batched.  p.groups = batch count (>= 1).
template <class T, int EPI>
int launch_gemm16(Gemm16Params p, hipStream_t s) {
  const int dsz = (EPI == EPI_F32) ? 4 : 2;
  // (32-bit per-lane byte offsets inside a tile bound the leading dimensions)
  const bool vec = (p.K % 8 == 0) && (p.N % 8 == 0) && (p.lda % 8 == 0) && (p.ldb % 8 == 0) &&
                   (p.lda < (1L << 21)) && (p.ldb < (1L << 21)) &&
                   ((p.ldd * dsz) % 16 == 0) && (p.strideA % 8 == 0) && (p.strideB % 8 == 0) &&
                   ((p.strideD * dsz) % 16 == 0) && aligned16(p.A) && aligned16(p.B) && aligned16(p.D) &&
                   (!p.bias || aligned16(p.bias));
  if (!vec) {
    // few rows: the streaming kernel reads B where it lies
    if (p.groups == 1 && p.M <= kLooseMaxM && p.N >= 8 && few_rows16_in_range(p.M, p.N, p.K, p.lda, p.ldb)) {
      const int rc = launch_gemm16_skinny<T, EPI>(p, skinny_loose_splits(p.N, p.K), true, s);
      if (rc != kNoScratch) return rc;
    }
    // small products go one thread per output element; above about 2^24 multiply-adds the
    // copies into aligned buffers cost less than that kernel loses
    if ((double)p.M * p.N * p.K * p.groups >= (double)(1L << 24) && p.M >= 16 && p.N >= 16 &&
        p.K + 8 < (1L << 21) && p.N + 8 < (1L << 21))
      return launch_gemm16_repitched<T, EPI>(p, s);
    dim3 block(32, 8), grid(ceil_div(p.N, 32), ceil_div(p.M, 8), p.groups);
    hipLaunchKernelGGL((gemm16_generic_kernel<T, EPI>), grid, block, 0, s, p);
    return launch_status();
  }
  Gemm16Schedule sch = select_gemm16_schedule(p.M, p.N, p.K, p.groups);
  // The f32 partials of a K split lie in the stream's workspace; without one of their size (a capture on a stream with none or a smaller one, a full
  // device) K stays whole on the same tiles.
  float* ws = nullptr;
  if (!sch.skinny && (sch.split_k > 1 || sch.rest_split > 1)) {
    const size_t rest = (size_t)ceil_div(p.M, 256) * ceil_div(p.N, 256) % 256;
    const size_t floats = sch.split_k > 1 ? (size_t)p.M * p.N * sch.split_k : rest * sch.rest_split * 256 * 256;
    ws = static_cast<float*>(stream_workspace_or_null(s, floats * sizeof(float)));
    if (!ws) sch.split_k = sch.rest_split = 1;
  }
  // bias / activation: the tile kernels have a separate instantiation for it (f32 out)
  const bool fused = p.bias != nullptr || p.act != ACT_NONE;
  if constexpr (EPI != EPI_F32) {
    if (fused) return kBadShape;
  }
  if (sch.tile == 256 && sch.tile_m == 128 && sch.split_k == 1) {
    if constexpr (EPI == EPI_F32) {
      if (fused) return launch_gemm16_tile<T, 128, 256, 2, 2, EPI_F32_FUSED, false, kBigTileMfma>(p, s);
    }
    return launch_gemm16_tile<T, 128, 256, 2, 2, EPI, false, kBigTileMfma>(p, s);
  }
  if (sch.tile == 256 && sch.split_k == 1) {
    const int tiles = ceil_div(p.M, 256) * ceil_div(p.N, 256);
    const int main_wgs = sch.rest_split > 1 ? tiles / 256 * 256 : 0;     // 0: every tile in one launch
    int rc = kOk;
    if (EPI == EPI_F32 && fused) {
      if constexpr (EPI == EPI_F32)
        rc = sch.pieces > 1 ? launch_gemm16_pieces<T, EPI_F32_FUSED>(p, sch.pieces, s)
                            : launch_gemm16_tile<T, 256, 256, 2, 2, EPI_F32_FUSED, false, kBigTileMfma>(p, s, main_wgs);
    } else {
      rc = sch.pieces > 1 ? launch_gemm16_pieces<T, EPI>(p, sch.pieces, s)
                          : launch_gemm16_tile<T, 256, 256, 2, 2, EPI, false, kBigTileMfma>(p, s, main_wgs);
    }
    if (rc != kOk || sch.rest_split <= 1) return rc;
    return launch_gemm16_rest<T, EPI>(p, main_wgs, tiles - main_wgs, sch.rest_split, ws, s);
  }
  const bool t128 = sch.tile == 128;
  if (sch.skinny) return launch_gemm16_skinny<T, EPI>(p, sch.split_k, false, s);
  // Every K split is one "batch" of the same kernel writing f32 partials, summed in
  // split order by a second kernel, so the result does not depend on scheduling.
  {
    const int splits = sch.split_k;
    if (splits > 1) {
      const size_t mn = (size_t)p.M * p.N;
      Gemm16Params q = p;
      q.K = split_steps(p.K, splits) * G16_BK;
      q.k_total = p.K;
      q.groups = splits;
      q.strideA = q.K;                       // split z reads A[:, z Ks ..) and B[z Ks .., :)
      q.strideB = (long)q.K * p.ldb;
      q.D = ws;
      q.bias = nullptr;                      // the epilogue runs once, on the summed partials
      q.act = ACT_NONE;
      q.ldd = p.N;
      q.strideD = (long)mn;
      const int rc =
          sch.tile == 256 && sch.tile_m == 128 ? launch_gemm16_tile<T, 128, 256, 2, 2, EPI_F32, false, kBigTileMfma>(q, s)
          : sch.tile == 256 ? launch_gemm16_tile<T, 256, 256, 2, 2, EPI_F32, false, kBigTileMfma>(q, s)
          : t128      ? launch_gemm16_tile<T, 128, 128, 2, 2, EPI_F32, false>(q, s)
                      : launch_gemm16_tile<T, 64, 64, 2, 2, EPI_F32, false>(q, s);
      if (rc == kOk) return launch_splitk_reduce<T, EPI>(ws, p.N, p, splits, 1, s);
      return rc;
    }
  }
  if constexpr (EPI == EPI_F32) {
    if (fused) {
      if (t128) return launch_gemm16_tile<T, 128, 128, 2, 2, EPI_F32_FUSED, false>(p, s);
      return launch_gemm16_tile<T, 64, 64, 2, 2, EPI_F32_FUSED, false>(p, s);
    }
  }
  if (t128) return launch_gemm16_tile<T, 128, 128, 2, 2, EPI, false>(p, s);
  return launch_gemm16_tile<T, 64, 64, 2, 2, EPI, false>(p, s);
}

// D[i] = act(G[i]) * U[i], four elements per thread (n % 4 == 0, 16-byte aligned pointers).
template <int ACT_DYNAMIC = 1>   // (a template so that every translation unit may include this header)
__global__ __launch_bounds__(256) void gate_mul_kernel(float* __restrict__ D, const float* __restrict__ G,
                                                       const float* __restrict__ U, long n4, int act) {
  const long i = (long)blockIdx.x * 256 + threadIdx.x;
  if (i >= n4) return;
  const float4 g = reinterpret_cast<const float4*>(G)[i], u = reinterpret_cast<const float4*>(U)[i];
  reinterpret_cast<float4*>(D)[i] =
      make_float4(activate(g.x, act) * u.x, activate(g.y, act) * u.y, activate(g.z, act) * u.z, activate(g.w, act) * u.w);
}

// Dense gated product D f32 = act(A Wg) * (A Wu); p.B = Wg, p.B2 = Wu, p.N = H.
template <class T>
int launch_gemm16_gated(Gemm16Params p, hipStream_t s) {
  // Few rows: both products are bound by reading their weight matrix once, which the dense
  // launcher's decode schedules (small tiles, K split over the chip) do at several times the rate
  // of one 256-row tile per 128 output columns.  Two products into stream-ordered scratch, then
  // the gate.
  if (p.M <= kWeightStreamMaxM && p.N % 8 == 0 && p.K % 8 == 0 && p.ldd == p.N && aligned16(p.D) &&
      (long)p.M * p.N >= 128L * 128L) {
    const size_t mn = (size_t)p.M * p.N;
    float* tmp = nullptr;
    if (!device_malloc_async(reinterpret_cast<void**>(&tmp), 2 * mn * sizeof(float), s)) return kDeviceFailed;
    Gemm16Params q = p;
    q.B2 = nullptr;
    q.act = ACT_NONE;
    q.bias = nullptr;
    q.groups = 1;
    q.strideA = q.strideB = q.strideD = 0;
    q.D = tmp;
    int rc = launch_gemm16<T, EPI_F32>(q, s);
    if (rc == kOk) {
      q.B = p.B2;
      q.D = tmp + mn;
      rc = launch_gemm16<T, EPI_F32>(q, s);
    }
    if (rc == kOk) {
      hipLaunchKernelGGL(gate_mul_kernel<1>, dim3((unsigned)((mn / 4 + 255) / 256)), dim3(256), 0, s,
                         static_cast<float*>(p.D), tmp, tmp + mn, (long)(mn / 4), p.act);
      rc = launch_status();
    }
    if (hipFreeAsync(tmp, s) != hipSuccess) { (void)hipGetLastError(); rc = rc == kOk ? kDeviceFailed : rc; }
    return rc;
  }
  const bool vec = (p.K % 8 == 0) && (p.N % 8 == 0) && (p.lda % 8 == 0) && (p.ldb % 8 == 0) &&
                   (p.lda < (1L << 21)) && (p.ldb < (1L << 21)) && (p.ldd % 4 == 0) && aligned16(p.A) &&
                   aligned16(p.B) && aligned16(p.B2) && aligned16(p.D);
  if (!vec || (long)p.M * p.N < 128L * 128L) {
    dim3 block(32, 8), grid(ceil_div(p.N, 32), ceil_div(p.M, 8), 1);
    hipLaunchKernelGGL((gemm16_generic_kernel<T, EPI_GATED_F32>), grid, block, 0, s, p);
    return launch_status();
  }
  return launch_gemm16_tile<T, 256, 256, 4, 1, EPI_GATED_F32, false, kBigTileMfma>(p, s);
}

// Grouped.  p.M = total rows S, p.groups = E, p.offsets = device int32[E+1].
template <class T, int EPI>
int launch_gemm16_grouped(Gemm16Params p, hipStream_t s) {
  const int dsz = (EPI == EPI_F32) ? 4 : 2;
  // (32-bit per-lane byte offsets inside a tile bound the leading dimensions)
  const bool vec = (p.K % 8 == 0) && (p.N % 8 == 0) && (p.lda % 8 == 0) && (p.ldb % 8 == 0) &&
                   (p.lda < (1L << 21)) && (p.ldb < (1L << 21)) &&
                   ((p.ldd * dsz) % 16 == 0) && (p.strideB % 8 == 0) && aligned16(p.A) &&
                   aligned16(p.B) && aligned16(p.D) && (EPI != EPI_SWIGLU16 || aligned16(p.B2));
  if (!vec) {
    dim3 block(32, 8), grid(ceil_div(p.N, 32), ceil_div(p.M, 8), 1);
    hipLaunchKernelGGL((gemm16_grouped_generic_kernel<T, EPI>), grid, block, 0, s, p);
    return launch_status();
  }
  // groups that average at most a tile of rows (a chunk of a thousand tokens over 64 experts): see MID at the kernel
  const bool mid = (long)p.M <= 256L * p.groups;
  // Weights that outgrow the memory-side cache are streamed past it while their panels are read by one row tile: groups
  // that average at most 240 rows.  Closer to the tile's 256 half of the groups have a second tile, whose reads then miss (the
  // whole layer with the hint / without: 64 experts of 4096 x 1408, 64 tokens 357 / 393 us, 1024 500 / 520, 1840, 230 rows a
  // group, 576 / 613, 2048, 256 rows, 793 / 756; 8 experts of 4096 x 4096, 920 tokens 236 / 239, 1024 318 / 295).
  const bool nt = (long)p.M <= 240L * p.groups &&
                  (EPI == EPI_SWIGLU16 ? 4.0 : 2.0) * p.K * p.N * p.groups >= kStreamOnceBytes;
  if constexpr (EPI == EPI_SWIGLU16) {
    if (mid && nt) return launch_gemm16_tile<T, 256, 256, 2, 2, EPI, true, kGroupedTileMfma, true, true>(p, s);
    if (mid) return launch_gemm16_tile<T, 256, 256, 2, 2, EPI, true, kGroupedTileMfma, true>(p, s);
    return launch_gemm16_tile<T, 256, 256, 2, 2, EPI, true, kGroupedTileMfma>(p, s);
  } else {
    if ((long)p.M < 64L * p.groups) {
      if (nt) return launch_gemm16_tile<T, 128, 128, 2, 2, EPI, true, 32, false, true>(p, s);
      return launch_gemm16_tile<T, 128, 128, 2, 2, EPI, true>(p, s);
    }
    if (mid && nt) return launch_gemm16_tile<T, 256, 256, 2, 2, EPI, true, kGroupedTileMfma, true, true>(p, s);
    if (mid) return launch_gemm16_tile<T, 256, 256, 2, 2, EPI, true, kGroupedTileMfma, true>(p, s);
    return launch_gemm16_tile<T, 256, 256, 2, 2, EPI, true, kGroupedTileMfma>(p, s);
  }
}

}  // namespace tsr950
