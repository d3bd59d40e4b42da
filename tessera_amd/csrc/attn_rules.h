// Which attention forward kernel and division of its work a problem gets (host code, no device headers).
#pragma once
#include <algorithm>

namespace tsr950 {

// Key splits of the decode kernel at padded head dimensions (DP: 64, 128 or 256, the compiled one): the fewest steps
// of one wave, a tile of 32 keys (and 1.5 for a workgroup's start and end; for the merge of the splits 2, at DP 256 one, as its
// tiles take longer) over the rounds in which a compute unit, which holds two workgroups at DP 64 and one above, takes them.  At most about two workgroups per
// compute unit, at least two tiles for every wave of a split.  (Two workgroups per unit whatever it holds left a second
// round: D 80, 256 heads x 500 keys 21.4 us in two splits, 14.8 in one; 64 x 2048 21.9 in eight, 18.3 in four.)
inline int pad_splits(int DP, int kvheads, int tiles, int waves) {
  const int slots = DP <= 64 ? 512 : 256;
  const int most = std::max(1, std::min((512 + kvheads - 1) / kvheads, tiles / (2 * waves)));
  int best = 1;
  double best_steps = 1e30;
  for (int n = 1; n <= most; ++n) {
    const int per_wave = ((tiles + n - 1) / n + waves - 1) / waves;
    const long parts = (tiles + per_wave * waves - 1) / (per_wave * waves);
    const double steps = (double)((kvheads * parts + slots - 1) / slots) * (per_wave + 1.5) + (parts <= 1 ? 0.0 : DP <= 128 ? 2.0 : 1.0);
    if (steps < best_steps) { best_steps = steps; best = n; }
  }
  return best;
}

// One query head per KV head at head dimensions between 64 and 128: where the decode kernel's workgroups need twice the
// rounds of the general kernel's (which share a compute unit in pairs), the general one serves up to 1023 keys (D 80: 257 heads
// x 500 keys 27.4 us against 20.9, 512 x 64 11.3 / 9.5, 1024 x 250 35.0 / 30.5; but 768 x 500 40.4 / 44.5, 512 x 1000 43.5 /
// 43.4, 257 x 2048 61.7 / 65.1).
inline bool pad_general(int kvheads, int Sk, int D) {
  return D > 64 && D < 128 && Sk < 1024 && kvheads > 256 && (kvheads + 255) / 256 >= 2 * ((kvheads + 511) / 512);
}

// Workgroup size (8 waves: 256 query rows, 4: 128) and key splits of the plain forward kernel at DP <= 128.
struct FlashShape { int waves, nsplit; };
struct FlashProblem { int B, Hq, Hkv, Sq, Sk, D; bool bias; };

// Key splits of 8-wave workgroups of `rows` query rows: few workgroups against a long key range (a chunk of queries
// against a long context) get about two workgroups per compute unit, at least 8 tiles (512 keys) a split.
inline int split8(const FlashProblem& p, int rows) {
  const long wgs = (long)p.B * p.Hq * ((p.Sq + rows - 1) / rows);
  if (wgs >= 192 || p.bias) return 1;
  return (int)std::max<long>(1, std::min<long>(std::min<long>((512 + wgs - 1) / wgs, (p.Sk + 63) / 64 / 8), 64));
}

// The order of 4-wave workgroups: the query blocks last, all heads' heavy blocks first; head after head, as with 8 waves, where
// that order would read K and V from memory for every query block: 90 MB of them, no heads that share them, and more heads than
// leave two blocks of one in flight.  (Bf16, D 128, Hq = Hkv = 32, causal, blocks last / head after head / 8 waves: B 20 x S 360
// 94.7 / 79.9 / 85.7 us, B 16 x S 600 145 / 124 / 130, B 24 x S 640 220 / 185 / 195; but B 9 x S 512, 75 MB, 60.0 /
// 70.2 / 70.4, and 160 heads, 1592 rows on 1792 keys, 147 MB, 192 / 210 / 198.)
inline bool flash_blocks_last(const FlashProblem& p) {
  return p.Hq != p.Hkv || p.D <= 96 || p.B * p.Hkv < 300 || 4.0 * p.B * p.Hkv * p.Sk * p.D < 9.0e7;
}

// tiles_of(q0, rows): 64-key tiles that the query rows [q0, q0 + rows) walk.  Estimated in steps of a 256-row workgroup (one
// tile; 4 more for its start and end, 6 for a part of a split walk):
//   8 waves (256 rows): one workgroup per compute unit, the longest walk or the work over 256 units;
//   4 waves (128 rows): a step is 1.1 with a second workgroup on the unit (K and V tiles are loaded twice),
//   0.7 without; split walks are nearly equal, so their workgroups come in whole rounds; a split costs a merge, 6 steps.
// What it weighs: 128 rows waste less on ragged lengths and spread short or few sequences over more units, 256
// rows read K and V half as often.  Measured, 8 waves against 4 (bf16, D 128, Hq 32, Hkv 8, causal): B 2 x S 500
// 23.0 -> 19.1 us, B 1 x S 1000 37.3 (two splits) -> 28.0 (none), B 1 x S 2048 61.6 -> 54.9, B 9 x S 384 45.5 -> 37.1,
// 512 rows on 4096 keys 60.4 (8 splits) -> 50.8 (4); but 512 rows on 32768 282 -> 298, 1024 on 32768 517 -> 540,
// B 1 x S 4096 149 -> 162, and the same at more rows, which stay on 8 waves.  Over 1220 timed shapes the choice is more than 3 %
// behind 8 waves at twelve, eleven with 384 KV heads of one query head (B 12, S 300 to 640: 3 to 8 %), and ahead by up to a third.
template <class Tiles>
FlashShape flash_shape(const FlashProblem& p, Tiles tiles_of) {
  const long heads = (long)p.B * p.Hq;
  const FlashShape wide{8, split8(p, 256)};
  if (p.Sq > 8192 || heads * p.Sq > (1L << 22)) return wide;
  struct Walks { double longest, shortest, total; };
  auto walks = [&](int rows) {
    Walks w{0, 1e30, 0};
    for (int q0 = 0; q0 < p.Sq; q0 += rows) {
      const double n = tiles_of(q0, std::min(rows, p.Sq - q0));
      w.longest = std::max(w.longest, n);
      w.shortest = std::min(w.shortest, n);
      w.total += n * heads;
    }
    return w;
  };
  const long n8 = heads * ((p.Sq + 255) / 256), n4 = heads * ((p.Sq + 127) / 128);
  // 257 to 384 rows in one round of 8-wave workgroups: the second, half-empty one ends with the first, so three
  // blocks gain only while the third is small as well (Hq 32, Hkv 4, 8 / 4 waves: B 4 x S 300 17.2 / 16.3 us, 350 17.5 / 18.5; with
  // fewer heads only at padded head dimensions: D 80, B 1 x S 342 14.7 / 15.7).
  // The same with one block more at those (D 80, B 10 x Hq 8 x S 640 22.5 / 25.1; S 512 22.4 / 20.5, 800 28.4 / 26.1).
  const bool padded = p.D > 64 && p.D < 128, half_block = (p.Sq - 1) % 256 < 128;
  if (p.Sq > 320 && p.Sq <= 384 && n8 <= 256 && (n4 > 256 || padded)) return wide;
  if (padded && half_block && p.Sq > 256 && p.Sq <= 640 && n8 <= 256 && n4 > 256) return wide;
  // One 8-wave block but two of 4, heads that share no K and V, 45 MB and more: they are read twice from memory (S 256, 32
  // heads, B 16 39.3 / 46.0 us; up to 42 MB, B 10, 35.4 / 34.0).
  const double kv_bytes = p.Hq <= 2 * p.Hkv && p.D > 64 ? 512.0 * p.B * p.Hkv * p.Sk : 0.0;
  if (p.Sq > 128 && p.Sq <= 256 && n4 > 512 && kv_bytes > 4.5e7) return wide;
  const Walks w8 = walks(256), w4 = walks(128);
  // (walks under 48 tiles: what a split adds shows less, and the splits of 8 waves, 512 keys each, gain nothing beside
  // one block: 227 rows on 1127 keys 29.5 us with them, 26.2 in 4 waves; nor do they where the walks are far from equal: D 80,
  // Hq 8, S 3065 54.8 us with them, 49.5 in 4 waves)
  const bool short_walks = w8.longest < 48, unequal = w8.longest > 4 * w8.shortest;
  auto ends = [&](int n) { return n > 1 && !short_walks ? 6.0 : 4.0; };
  auto merge = [](int n) { return n > 1 ? 6.0 : 0.0; };
  auto rounds = [](long wgs, int slots) { return (double)((wgs + slots - 1) / slots); };
  // (one block of at most 128 rows keeps half of eight waves busy, one of 192 six)
  const double few = p.Sq <= 128 ? 0.68 : p.Sq <= 192 ? 0.75 : 1.0;
  auto t8 = [&](int n) {
    const double longest = w8.longest / n + ends(n), shortest = w8.shortest / n + ends(n);
    const double all = (w8.total + n8 * n * ends(n)) / 256;
    if (n8 * n <= 256) return few * longest + merge(n);
    if (n > 1) return std::max({longest, shortest * rounds(n8 * n, 256), all}) + merge(n);
    return std::max(longest, all + 0.5 * shortest);
  };
  auto t4 = [&](int n) {
    const double longest = w4.longest / n + ends(n), shortest = w4.shortest / n + ends(n);
    const double all = (w4.total + n4 * n * ends(n)) / 512 + 0.5 * shortest;
    if (n4 * n <= 256) return 0.7 * longest + merge(n);
    if (n4 * n <= 512) return 1.1 * shortest + 0.7 * (longest - shortest) + merge(n);
    if (n > 1) return 1.1 * std::max({longest, shortest * rounds(n4 * n, 512), all}) + merge(n);
    // (heads that no XCD owns share no L2, and the second read of K and V then costs more: B 13 x Hq 32 x Hkv 4 x S 591
    // 101 -> 106 us)
    return (p.B * p.Hkv % 8 ? 1.35 : 1.1) * std::max(longest, all);
  };
  int best = 1;
  // (from 192 blocks on never: a split takes the stream's workspace, which a captured call must find allocated)
  const int most = n8 >= 192 ? 1 : (int)std::min<long>(std::min<long>(std::max<long>(512 / n4, 1), (p.Sk + 63) / 64 / 8), 64);
  for (int n = 2; n <= most; ++n)
    if (t4(n) < t4(best)) best = n;
  // (splits of short walks that put two workgroups on a unit are no better than 8 waves and theirs: B 1 x Hq 8 x
  // Hkv 8 x S 2048 36.8 us against 35.4)
  if (best > 1 && n4 * best > 256 && w4.longest < 48) return wide;
  // (129 to 192 rows leave 8 waves' splits nearly as good: 180 rows on 1080 keys 25.9 / 29.4)
  const double margin = best > 1 && !short_walks && !unequal ? 1.0 : p.Sq > 128 && p.Sq <= 192 && wide.nsplit > 1 ? 1.08 : 1.03;
  return margin * t4(best) < t8((short_walks && p.Sq > 192) || unequal ? 1 : wide.nsplit) ? FlashShape{4, best} : wide;
}

}  // namespace tsr950
