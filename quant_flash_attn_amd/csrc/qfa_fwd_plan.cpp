// Into how many parts the keys of the INT8-score forward are split (qfa_fwd.hip, qfa_fwd_wide.hip).
#include <algorithm>

#include "qfa_host.h"

namespace qfa {

// A workgroup of 128 queries is a chain of 64-key tiles whose pace hardly depends on what the rest of the chip does, so few
// queries over many keys take the time of one chain while the other CUs idle (4 heads, 333 queries, 30000 keys of 128:
// 12 workgroups, 458 us; their keys in 20 parts 40 us, with the merge).  A second workgroup on a CU is only worth a third to a
// half of one more CU, and each part writes its O in fp32 for the merge to read.  The model below is that and no more; its
// constants are fitted to 2600 shapes of 1 to 512 heads, 17 to 16384 queries, 64 to 30000 keys, causal or not, each timed with
// every division of its keys.  Where splitting can help it takes the logarithmic mean over the shapes from 1.9 to 1.01 of the
// best division's time.  Gains of less than 5 % are left, being within the model's error: no shape got slower by
// more than 4 %.
struct FwdCost {
  double tile[3];      // us per tile with one, two, three workgroups on a CU
  int resident;        // workgroups on a CU
  double start, tail;  // of a workgroup, in tiles; share of the last workgroup that runs alone
  double merge, mb;    // us: the merge, and per MB that it moves
  double base;
};

static const FwdCost &fwd_cost(int D) {
  static const FwdCost c64 = {{0.85, 1.00, 1.34}, 3, 1.85, 0.28, 2.1, 0.275, 4.3}, c128 = {{1.13, 1.45, 1.45}, 2, 1.14, 0.48, 2.6, 0.265, 4.5},
                       c256 = {{1.58, 1.58, 1.58}, 1, 1.08, 0.53, 4.1, 0.26, 5.2};
  return D == 64 ? c64 : D == 128 ? c128 : c256;
}

void fwd_plan(int64_t BH, int64_t Nq, int64_t Nk, int D, int causal, int *splits, int *keys_per_split) {
  constexpr int64_t MAX_WGS = 1700, MAX_SPLITS = 64;
  const FwdCost &c = fwd_cost(D);
  const int64_t tiles = (Nk + 63) / 64, mblocks = (Nq + 127) / 128, coff = Nk - Nq;
  auto cost = [&](int64_t s, int64_t each) {
    int64_t total = 0, wgs = 0, longest = 0;   // tiles of a head; its workgroups that have any; those of the longest
    for (int64_t mb = causal ? 0 : mblocks - 1; mb < mblocks; ++mb) {
      const int64_t seen = causal ? (std::min(Nk, (mb + 1) * 128 + coff) + 63) / 64 : tiles;
      total += seen;
      wgs += (seen + each - 1) / each;
      longest = std::max(longest, std::min(each, seen));
    }
    const int64_t heads = causal ? BH : BH * mblocks, n = wgs * heads, slots = 256 * c.resident;
    const double last = (double)longest + c.start;
    const double body = n <= slots ? last * c.tile[(n + 255) / 256 - 1]
                                   : ((total * heads + n * c.start) / slots + c.tail * last) * c.tile[c.resident - 1];
    return c.base + body + (s > 1 ? c.merge + c.mb * 8e-6 * (double)(BH * Nq * s * (D + 2)) : 0.0);
  };
  int64_t best_each = tiles;
  const int64_t most = BH <= MAX_WGS && mblocks <= MAX_WGS ? std::min(std::min(tiles, MAX_SPLITS), MAX_WGS / (BH * mblocks)) : 0;
  if (most > 1) {
    double best = 0.95 * cost(1, tiles);
    for (int64_t s = 2; s <= most; ++s) {
      const int64_t each = (tiles + s - 1) / s;
      if ((tiles + each - 1) / each != s) continue;
      const double t = cost(s, each);
      if (t < best) {
        best = t;
        best_each = each;
      }
    }
  }
  *splits = (int)((tiles + best_each - 1) / best_each);
  *keys_per_split = (int)best_each * 64;
}

int64_t fwd_workspace_bytes(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int D, int causal) {
  int splits, keys;
  fwd_plan(B * H, Nq, Nk, D, causal, &splits, &keys);
  return splits > 1 ? B * H * Nq * splits * (int64_t)(D + 2) * 4 : 0;
}

}  // namespace qfa
