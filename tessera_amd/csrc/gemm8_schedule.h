// Tile and K-split choice of the 8-bit GEMM (int8 / e4m3) for an aligned problem: the one place the
// decision lives (the launcher and the schedule query of the C ABI both call it).  Host code only.
#pragma once
#include <algorithm>
#include <cmath>

namespace tsr950 {

struct Gemm8Schedule {
  int tile_m;    // rows of the workgroup tile: 256 or 128 (tile kernel), 32 or 64 (few-row streaming kernel)
  int tile_n;    // columns: 256 (tile kernel) or 128 (streaming kernel's strip)
  int tile_k;    // bytes of K per step: 128 (tile kernel) or 64 (a streaming slice)
  int split_k;   // K slices summed by the split-sum kernel (1 = none)
  bool skinny;   // the few-row streaming kernel
};

constexpr int kGemm8SkinnyMaxM = 64;

// Time estimate (microseconds) of `tiles` workgroup tiles of bm x 256 walking `ksteps` 128-deep K steps,
// fitted to timings of both tiles on this part over products from 1024^3 to 8192^3: rounds of 256
// concurrent tiles; a tile's cost outside its K loop grows with the number of tiles storing at once, and
// a K step is slower with every compute unit busy (the board's power limit sets the clock).
inline double est_tiles8_us(int bm, long tiles, int ksteps) {
  const double f0 = bm == 256 ? 9.6 : 6.0, f1 = 3.0, s0 = bm == 256 ? 1.2 : 0.62, s1 = bm == 256 ? 0.48 : 0.30;
  const long full = tiles / 256, rem = tiles % 256;
  double t = (double)full * (f0 + f1 + ksteps * (s0 + s1));
  if (rem) t += f0 + f1 * rem / 256.0 + ksteps * (s0 + s1 * std::min(1.0, std::max(0.0, (rem - 144) / 112.0)));
  return t;
}

// Waves in a workgroup of the streaming kernel: 8 up to 32 rows, 4 above (twice the accumulators).  loose: four up to 32
// rows, too.  Off the 128-byte grid a row's piece lies in two cache lines and neighbouring strips want the same line, and eight
// waves with a workgroup's whole K range in flight read at half the rate (16 rows, N 8191 x K 4097: 65 us with
// eight, 28 with four, 47 by copies into aligned buffers; 14335 x 2049 79, 35 and 41).  Up to one slice for each of
// eight waves (K 512), eight: 16 x 1003 x 259 9.8 against 11.3.
inline int gemm8_skinny_waves(int M, int K, bool loose) { return M <= 32 && (!loose || K <= 512) ? 8 : 4; }

// Time estimate (microseconds) of the streaming kernel, fitted (9 % rms) to forced splits over 17 weight shapes (512 to
// 8192 columns, 1536 to 14336 rows) under 1 to 64 rows: a launch; a workgroup's rows of B, each 2.1 ns where it is alone
// (eight waves; 4.5 with four, whose accumulators hold two row blocks) and 6.5 (7.5) beside 255 others, in rounds of 256;
// a million results (with K in several parts: partials) 2.5 us, and a second launch, 1.5 us, to sum the parts.
inline double est_stream8_us(int waves, int M, int N, int K, int splits) {
  const long wgs = (long)((N + 127) / 128) * splits;
  const double full = (double)std::min(wgs, 256L) / 256.0;
  const double row_ns = waves == 8 ? 2.1 + 4.4 * full : 4.5 + 3.0 * std::sqrt(full);
  const double rows = ((K + splits - 1) / splits + 63) / 64 * 64.0;
  return 3.4 + row_ns * 1e-3 * rows * (double)((wgs + 255) / 256) + 2.5e-6 * M * N * splits + (splits > 1 ? 1.5 : 0.0);
}

// K splits of the streaming kernel by that estimate: never over one workgroup per compute unit (the second round
// would be nearly empty), at least one 64-row slice for each of its waves.  (Without the partials in the estimate every
// short product was split as far as it went: 64 x 1024 x 8192 in 32 parts 14.2 us, in 16 11.8; 32 x 2048 x 8192 16 / 8
// parts 11.3 / 10.1.)
inline int gemm8_skinny_splits(int waves, int M, int N, int K) {
  const int strips = (N + 127) / 128;
  const int most = std::max(1, std::min(256 / strips, K / (waves * 64)));
  int best = 1;
  double best_us = 1e30;
  for (int splits = 1; splits <= most; ++splits) {
    const double us = est_stream8_us(waves, M, N, K, splits);
    if (us < best_us) { best_us = us; best = splits; }
  }
  return best;
}

// Time estimate (microseconds) of the tiles for up to 1024 rows against a weight matrix that streams from HBM,
// fitted (10 % rms) to forced schedules on this part — the 128- and 256-row tiles, K in 1 to 32 parts, 18 weight
// shapes from 2048 x 7168 to 32768 x 4096 (the weights cycled through copies) under 16 to 1024 rows: a launch cost, then the
// larger of the busiest compute unit's K steps (its first workgroup at `step`, every further one sharing the unit at
// `shared` per step) and the time to stream the tile columns of B at `tbs` TB/s, which takes about
// 155 workgroups in flight to reach and is stretched by a last, partly filled round; the sum over
// K parts adds 2 us and 1.4 us per million partials.
struct Gemm8Fit { double launch, step, shared, tbs; };
constexpr Gemm8Fit kGemm8Fit[2] = {{6.51, 0.780, 1.121, 6.52},     // 128 x 256 tiles (a step = 128 of K)
                                   {9.82, 1.107, 1.944, 5.31}};    // 256 x 256 tiles
inline double est_gemm8_fit_us(int tile_m, int M, int N, int K, int splits) {
  const Gemm8Fit& f = kGemm8Fit[tile_m == 256];
  const long cols = (N + 255) / 256, wgs = (M + tile_m - 1) / tile_m * cols * splits;
  const double steps = (double)K / 128 / splits;
  const double busiest = (double)((wgs + 255) / 256);
  const double compute = steps * (f.step + f.shared * (busiest - 1.0));
  const double bytes = (double)K * cols * 256;
  const double stream = bytes / (f.tbs * 1e6 * std::min(1.0, wgs / 155.0)) * (wgs > 256 ? busiest * 256.0 / wgs : 1.0);
  const double sum = splits > 1 ? 2.06 + (double)M * N * splits * 1.43e-6 : 0.0;
  return f.launch + std::max(compute, stream) + sum;
}

// The rule: the streaming kernel for few rows, else tile rows and a power-of-two K split by est_tiles8_us.
inline Gemm8Schedule select_gemm8_rule(int M, int N, int K) {
  auto cdiv = [](long a, long b) { return (a + b - 1) / b; };
  // At most 64 rows (quantised decode): the streaming kernel.  (Below 1024 rows of B the tiles are as good:
  // 48 x 4096 x 512 10.2 us against 12.3.)
  if (M <= kGemm8SkinnyMaxM && K % 16 == 0 && K >= 1024) {
    const int kps = (int)cdiv(cdiv(K, gemm8_skinny_splits(gemm8_skinny_waves(M, K, false), M, N, K)), 64) * 64;
    return {M <= 32 ? 32 : 64, 128, 64, (int)cdiv(K, kps), true};
  }
  // Tile rows (256 or 128) and K slices by estimated time.  Few tiles and a long K (few rows against a
  // big weight matrix): K is split over the idle compute units (a power of two, tiles x slices within
  // the 256 compute units, every slice at least 512 deep); the sum over the slices reads the partials
  // and writes the result at about 4.4 TB/s.
  const int ksteps = (int)cdiv(K, 128);
  const long tn = cdiv(N, 256);
  Gemm8Schedule best{256, 256, 128, 1, false};
  double best_us = 1e30;
  for (int cand : {256, 128}) {
    const long tiles = cdiv(M, cand) * tn;
    const double us1 = est_tiles8_us(cand, tiles, ksteps);
    if (us1 < best_us) { best_us = us1; best.tile_m = cand; best.split_k = 1; }
    if (tiles <= 128)
      for (int sp = 2; sp <= 16 && tiles * sp <= 256 && K / sp >= 512; sp *= 2) {
        const double us = est_tiles8_us(cand, tiles * sp, (int)cdiv(ksteps, sp)) + 2.0 +
                          (double)M * N * (4.0 * sp + 4.0) / 4.4e6;
        if (us < best_us) { best_us = us; best.tile_m = cand; best.split_k = sp; }
      }
  }
  return best;
}

// The schedule of an aligned 8-bit product: the rule above, unless — for 16 to 1024 rows under a weight
// matrix of the sizes the fits cover — the estimate of a tile schedule is well below that of the rule's: by a tenth,
// the fits' own error, and where the rule is the streaming kernel, whose estimate comes from timings of its own, by 13 %
// up to 32 rows (32 x 128256 x 2048, 20 % below: tiles 55.8 us, the streaming kernel 62.4) and by 18 % above (64 x 8192 x 8192,
// 11 % below: 25.6 against 24.7; 64 x 28672 x 4096, 17 %: 39.6 against 35.1).  Its split is the best by its estimate already.
inline Gemm8Schedule select_gemm8_schedule(int M, int N, int K) {
  const Gemm8Schedule rule = select_gemm8_rule(M, N, K);
  if (!(M >= 16 && M <= 1024 && N >= 2048 && K >= 1024)) return rule;
  const double rule_us = rule.skinny ? est_stream8_us(gemm8_skinny_waves(M, K, false), M, N, K, rule.split_k)
                                     : est_gemm8_fit_us(rule.tile_m, M, N, K, rule.split_k);
  Gemm8Schedule best = rule;
  double best_us = (!rule.skinny ? 0.9 : M <= 32 ? 0.87 : 0.82) * rule_us;
  for (int tile_m : {128, 256})
    for (int sp : {1, 2, 3, 4, 5, 6, 7, 8, 12, 16}) {
      if (K / sp < 512) continue;
      // (up to 32 rows a tile has to beat the streaming kernel by another 5 %: below the 16 rows the fit
      // starts at, that kernel is the faster by more)
      const double us = est_gemm8_fit_us(tile_m, M, N, K, sp) * (M <= 32 ? 1.05 : 1.0);
      if (us >= best_us) continue;
      best_us = us;
      best = Gemm8Schedule{tile_m, 256, 128, sp, false};
    }
  return best;
}

}  // namespace tsr950
