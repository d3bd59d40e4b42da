// Which attention forward kernel and division of its work a problem gets (host code, no device headers).
#pragma once
#include <algorithm>
#include <vector>

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

}  // namespace tsr950
