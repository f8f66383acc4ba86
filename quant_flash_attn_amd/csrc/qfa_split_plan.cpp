// Into how many parts the streamed rows of the INT8-score kernels are dealt: the keys of the forward (qfa_fwd.hip,
// qfa_fwd_wide.hip) and of dQ (qfa_bwd_dq.inc), the queries of dK and dV (qfa_bwd_dkv.inc).
//
// A workgroup is a chain of tiles whose pace hardly depends on what the rest of the chip does, so few rows against many take the
// time of one chain while the other CUs idle (forward, 4 heads, 333 queries, 30000 keys of 128: 12 workgroups, 458 us; their
// keys in 20 parts 40 us, with the merge).  A second workgroup on a CU is only worth a third to a half of one more CU, and each
// part writes its fp32 results for another kernel to add.  The model below is that and no more.  Its constants are fitted to
// 2600 (forward) and 1000 (backward) shapes of 1 to 512 heads, 17 to 16384 queries, 64 to 30000 keys, causal or not, each timed
// with every division.  Over these shapes the forward takes 1.01 times the best division's time in the geometric mean where the
// undivided one takes 1.9 times, dK / dV 1.01 against 1.045, dQ 1.004 against 1.11 (both of the whole backward).  Small gains
// are left, being within the model's error: of 1500 more backwards that are divided (0.63 times the undivided time in the geometric
// mean) three take more than 1.06 times, 1.12 at most; forwards up to 1.04.
#include <algorithm>
#include <cmath>

#include "qfa_host.h"

namespace qfa {

struct SplitCost {
  double tile[3];      // us per tile with one, two, three workgroups on a CU
  int resident;        // workgroups on a CU
  double start, tail;  // of a workgroup, in tiles; share of the last workgroup that runs alone
  double merge, mb;    // us: the merge or sum, and per MB that it moves
  double base;
};

constexpr int64_t MAX_WGS = 1700, MAX_WGS_BWD = 1100;   // of a divided launch: as far as was measured
// Of the parts of one launch: what MAX_WGS leaves of the forward (214 MiB, long sequences of few wide heads; 192 MiB cost 3 heads,
// 22757 x 22757 of 256, causal, 1019 -> 1474 us), and less than dK and dV could fill (275 MiB).  Between 1.03 times faster and slower
// where it bites there (5 heads of 17926 of 128, forward and backward: 3168 -> 3077 us; 5 of 24880, causal: 3680 -> 3765).
constexpr int64_t MAX_PART_FLOATS = QFA_SPLIT_PART_BYTES / 4;

// `blocks` workgroups of `rows` rows each for each of `heads` heads, the streamed rows in tiles of `tile` (64 or 32), s parts of
// `each` rows; ends: block i sees streamed rows up to (i + 1) * rows + coff, otherwise from i * rows - coff on.
// group_log2: how the backward's launches deal their blocks (-1: the forward's): every XCD takes an eighth of the blocks in a row
// with all their parts, causal those of 2^group_log2 heads in turn from the longest block on.  The first XCD then has most to
// do, and 255 workgroups of 85 blocks are 33 on its 32 CUs (5 heads, 4270 x 4270 of 128: counted evenly they were one round, and
// 259 us took the place of 218).
struct SplitWork {
  int64_t heads, blocks, rows, streamed, tile, coff;
  bool causal, ends;
  int group_log2 = -1;
  double total = 0, longest = 0;   // tiles of a head, of its longest block
  int64_t seen(int64_t i) const {
    if (!causal) return streamed;
    return ends ? std::min(streamed, (i + 1) * rows + coff) : streamed - std::max<int64_t>(i * rows - coff, 0);
  }
  void count() {   // (only for launches that may be divided: few blocks)
    if (!causal) {
      longest = (double)((streamed + tile - 1) / tile);
      total = longest * (double)blocks;
      return;
    }
    for (int64_t i = 0; i < blocks; ++i) {
      const double n = (double)((seen(i) + tile - 1) / tile);
      total += n;
      longest = std::max(longest, n);
    }
  }
  // workgroups of the first XCD that have something to do, and their tiles
  void first_xcd(int64_t s, int64_t each, double *live, double *tiles) const {
    const int64_t ids = (heads * blocks + 7) / 8;
    if (!causal) {
      *live = (double)(ids * s);
      *tiles = (double)ids * longest;
      return;
    }
    const int64_t group = std::min<int64_t>(heads, (int64_t)1 << group_log2);
    int64_t n = 0, t = 0;
    for (int64_t at = 0; at < ids;) {
      const int64_t i = at / group % blocks, seen_rows = seen(ends ? blocks - 1 - i : i), many = std::min(group, ids - at);
      n += many * std::min<int64_t>(s, (int)(seen_rows + each - 1) / (int)each);
      t += many * ((seen_rows + tile - 1) / tile);
      at += many;
    }
    *live = (double)n;
    *tiles = (double)t;
  }
  double time(const SplitCost &c, int64_t s, int64_t each, double mbytes) const {
    const double per = (double)(each / tile);
    double n, all;   // workgroups with something to do and their tiles, of the chip
    if (group_log2 < 0) {
      n = (double)(blocks * s);
      if (causal) n = std::min(n, total / per + 0.5 * (double)blocks);   // the others have nothing to do
      n *= (double)heads;
      all = total * (double)heads;
    } else {
      first_xcd(s, each, &n, &all);
      n *= 8.0;
      all *= 8.0;
    }
    const double slots = 256.0 * c.resident, last = std::min(longest, per) + c.start;
    const double body = n <= slots ? last * c.tile[std::min(c.resident, (int)std::ceil(n / 256.0)) - 1]
                                   : ((all + n * c.start) / slots + c.tail * last) * c.tile[c.resident - 1];
    return c.base + body + (s > 1 ? c.merge + c.mb * mbytes : 0.0);
  }
};

// the parts of `streamed` rows that cost least, at most `most`: f(s, rows of a part) in us, if below `best`
template <typename F> static void best_division(int64_t streamed, int64_t most, double best, int64_t *splits, int64_t *each, F f) {
  const int64_t tiles = (streamed + 63) / 64;
  for (int64_t s = 2; s <= std::min(tiles, most); ++s) {
    const int64_t e = (tiles + s - 1) / s;
    if ((tiles + e - 1) / e != s) continue;
    const double t = f(s, e * 64);
    if (t < best) {
      best = t;
      *splits = s;
      *each = e * 64;
    }
  }
}

void fwd_plan(int64_t BH, int64_t Nq, int64_t Nk, int D, int causal, int *splits, int *keys_per_split) {
  static const SplitCost c64 = {{0.85, 1.00, 1.34}, 3, 1.85, 0.28, 2.1, 0.275, 4.3}, c128 = {{1.13, 1.45, 0}, 2, 1.14, 0.48, 2.6, 0.265, 4.5},
                         c256 = {{1.58, 0, 0}, 1, 1.08, 0.53, 4.1, 0.26, 5.2};
  const SplitCost &c = D == 64 ? c64 : D == 128 ? c128 : c256;
  const int64_t blocks = (Nq + 127) / 128;
  int64_t s = 1, each = (Nk + 63) / 64 * 64;
  if (BH <= MAX_WGS && blocks <= MAX_WGS && 2 * BH * blocks <= MAX_WGS) {
    SplitWork w = {BH, blocks, 128, Nk, 64, Nk - Nq, causal != 0, true};
    w.count();
    best_division(Nk, std::min<int64_t>({64, MAX_WGS / (BH * blocks), MAX_PART_FLOATS / (BH * Nq * (D + 2))}), 0.92 * w.time(c, 1, each, 0), &s, &each,
                  [&](int64_t n, int64_t e) { return w.time(c, n, e, 8e-6 * (double)(BH * Nq * n * (D + 2))); });
  }
  *splits = (int)s;
  *keys_per_split = (int)each;
}

int64_t fwd_workspace_bytes(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int D, int causal) {
  int splits, keys;
  fwd_plan(B * H, Nq, Nk, D, causal, &splits, &keys);
  return splits > 1 ? B * H * Nq * splits * (int64_t)(D + 2) * 4 : 0;
}

// O past the caches where codes, V and O exceed the last-level one: else it pushes out what other workgroups read next, and where
// there are few keys its lines are still the cheaper to write.  29 calls of 256 to 2500 MiB, with and without a mask, the whole call
// (with a product that reads O behind it) against the same without the hint: head_dim 256 0.968 (0.984) of the time in the mean, 0.906 to
// 0.999 (0.963 to 0.998); 128 0.982 (0.994), 0.928 to 0.998 (0.979 to 1.016).  64 heads of 4096 x 256 causal 616 -> 579 us, 225 of 1525 x 572
// 327 -> 300, 256 of 4096 x 256 keys of 128 270 -> 251, 128 of 4096 x 128 causal 555 -> 544.  Below that size nothing is gained and the
// product loses (1024 of 300 x 128: 123 -> 123, 159 -> 163), and at head_dim 64 nothing was seen.  Rows that share their lines with those
// of other heads are written in pieces, which may take longer with the hint (1798 heads of 231 x 256, 266 -> 278 us)
bool fwd_o_once(int64_t BH, int64_t Nq, int64_t Nk, int D, const void *o, int64_t sob, int64_t soh, int64_t son) {
  return D >= 128 && BH * (Nq + Nk) * D * 3 > LAST_LEVEL_BYTES && rows_own_lines(o, sob, soh, son, 2 * D, 2);
}

// ---- backward
// Blocks of 32 rows per wave.  Two at head_dim 128: a step of 64 rows per wave costs 1 / 0.62 of one of 32, which need more LDS
// reads per row, but fill the chip with twice the workgroups and waste less of the last one (1024 x 1024, 16 heads: dQ 44 -> 22
// us; 2048 x 2048, 4 heads: 81 -> 36 us against 64 rows).  The cost of a launch on 256 CUs, one workgroup per CU, in steps of 32
// streamed rows: whole rounds when all are equally long; causal, the mean load and half of the longest, or the longest where
// all run at once (a tenth more, since the mean of shorter ones fills in better than that); starting and finishing a workgroup
// costs about two.  Both kernels' variants timed for 16 to 1024 heads of 64 to 2048 tokens: the choice is within 5 % of the
// best but for 128 heads of 768 (6 %); 256 heads of 200 and 256 causal tokens, the whole backward: 70 -> 66 and 74 -> 69 us with
// one round of 256-row workgroups.
static float undivided_cost(int64_t BH, int64_t rows, int64_t streamed, bool causal, float f, int rb, float step) {
  const int64_t nb = (rows + 128 * rb - 1) / (128 * rb);
  const float steps = (float)((streamed + 31) / 32) * step, fix = 2.0f;
  if (!causal) return (float)((nb * BH + 255) / 256) * (steps + fix);
  if (nb * BH <= 256) return 1.1f * (steps + fix);
  const float sum = (float)(nb * BH) * (steps * (1.0f - 0.5f * f) + 2.0f * (float)rb * step + fix);   // f: a head's triangle (trapezoid)
  return sum / 256.0f + 0.5f * steps;
}

// one of the two kernels: `tensors` fp32 results per row
static void bwd_part(int64_t BH, int64_t rows, int64_t streamed, int D, bool causal, bool ends, int64_t coff, float f, bool may_split,
                     const SplitCost (&c)[2], int tensors, int *blocks, int *splits, int *per_split) {
  int rb = 1;
  if (D == 128 && undivided_cost(BH, rows, streamed, causal, f, 1, 0.62f) >= undivided_cost(BH, rows, streamed, causal, f, 2, 1.0f)) rb = 2;
  int64_t s = 1, each = (streamed + 63) / 64 * 64;
  *blocks = rb;
  const int group_log2 = bwd_group_log2(streamed, D, ends);
  if (may_split && BH <= MAX_WGS_BWD && rows <= 128 * MAX_WGS_BWD) {
    SplitWork w[2];
    for (int r = 1; r <= (D == 128 ? 2 : 1); ++r) {
      w[r - 1] = {BH, (rows + 128 * r - 1) / (128 * r), 128 * r, streamed, 32, coff, causal, ends, group_log2};
      if (2 * BH * w[r - 1].blocks <= MAX_WGS_BWD || r == rb) w[r - 1].count();
    }
    const double undivided = w[rb - 1].time(c[rb - 1], 1, each, 0);
    double best = 0;
    for (int r = 1; r <= (D == 128 ? 2 : 1); ++r) {
      const SplitWork &x = w[r - 1];
      const int64_t was = s;
      // (with another number of rows per wave a division has to promise more: 12 heads of 4037, causal, promised 0.915, took 1.11)
      if (was == 1) best = (r == rb ? 0.93 : 0.9) * undivided;
      s = 1;
      const int64_t most = std::min<int64_t>({32, MAX_WGS_BWD / (BH * x.blocks), MAX_PART_FLOATS / (BH * rows * D * tensors)});
      best_division(streamed, most, best, &s, &each, [&](int64_t n, int64_t e) {
        return x.time(c[r - 1], n, e, 8e-6 * (double)(BH * rows * n) * D * tensors);
      });
      if (s > 1) {
        best = x.time(c[r - 1], s, each, 8e-6 * (double)(BH * rows * s) * D * tensors);
        *blocks = r;
      } else {
        s = was;
      }
    }
  }
  *splits = (int)s;
  *per_split = (int)each;
}

// ---- both kinds of workgroups in one launch (qfa_bwd_pair.h)
// Each kind by itself is planned above; together they leave less idle, so parts that fill the chip for one alone can be too many, and
// wide blocks too few no longer.  The estimate: where all workgroups run at once, the longest and a share of the mean load (they
// slow each other down); otherwise the mean load and what is left of the last dQ workgroup, or again the longest.  Fitted to 7100 shapes
// of 1 to 400 heads, 64 to 8192 keys, causal or not, with up to 29 divisions of both kinds each.  Only a division that it promises
// to be a tenth faster than the plan is taken: one call in nine, and of 2100 new ones (700 of a head_dim, timed as they are launched)
// it makes 0.90, 0.89 and 0.87 of the time in the mean (head_dim 64, 128, 256), 27 of them more than 1.04 times (1.14 at most: 3 heads,
// 31 x 357 of 256, 19.9 -> 22.6 us; 4 heads of 3917 x 128, 131 -> 147); taken whenever it is the fastest, 5 in a hundred of all calls
// at 128 would take more than 1.04 times.  8 heads of 1702 x 128 causal 73 -> 57 us, 2 x 1936 x 256 78 -> 56.
struct PairCost {
  double base, prep, sum, mb;   // us: launches; staging per MB (10^6 elements); the sum of parts and what it takes per MB
  double start[2], tail;        // of a workgroup of dK / dV and of dQ, in tiles; share of the last one that runs alone
  double tile[2][2];            // us per tile: [dK / dV, dQ][32, 64 rows per wave; at head_dim 64 one, two workgroups per CU]
  double crowd, over;           // of the mean load, added to the longest workgroup: within one round its share, beyond a fitted correction (below zero too)
};
constexpr int64_t SUM_BETWEEN = 128 << 20;   // of parts: more of both, and they are added between two launches
struct Share { int blocks, splits, each; double n, tiles, last, mbytes; };   // workgroups, tiles of all, of the longest

static double pair_time(const PairCost &c, int D, const Share &kv, const Share &q) {
  const double slots = D == 64 ? 512.0 : 256.0, n = kv.n + q.n;
  const double tk = c.tile[0][D == 64 ? n > 256.0 : kv.blocks - 1], tq = c.tile[1][D == 64 ? n > 256.0 : q.blocks - 1];
  const double ek = (kv.last + c.start[0]) * tk, eq = (q.last + c.start[1]) * tq, longest = std::max(ek, eq);
  const double mean = ((kv.tiles + kv.n * c.start[0]) * tk + (q.tiles + q.n * c.start[1]) * tq) / slots, mb = kv.mbytes + q.mbytes;
  const double body = n <= slots ? longest + c.crowd * mean : std::max(mean + c.tail * eq, longest + c.over * mean);
  return body + (mb > 0.0 ? c.sum + c.mb * mb : 0.0);
}

// divisions of one kind that are worth an estimate (`parts`: also those into more than one), the plan's own first; returns how many
constexpr int MAX_SHARES = 23;
static int shares(int64_t BH, int64_t rows, int64_t streamed, int D, bool causal, bool ends, int64_t coff, int tensors, bool parts, int blocks,
                  int splits, int each, Share *out) {
  static const int counts[] = {1, 2, 3, 4, 5, 6, 8, 10, 12, 16, 24};
  const int64_t tiles = (streamed + 63) / 64;
  int found = 0;
  SplitWork w;
  auto work = [&](int r) {
    w = {BH, (rows + 128 * r - 1) / (128 * r), 128 * r, streamed, 32, coff, causal, ends, bwd_group_log2(streamed, D, ends)};
    w.count();
  };
  auto add = [&](int r, int64_t s, int64_t e) {
    Share &x = out[found++];
    x.blocks = r; x.splits = (int)s; x.each = (int)e;
    w.first_xcd(s, e, &x.n, &x.tiles);
    x.n *= 8.0;
    x.tiles *= 8.0;
    x.last = std::min(w.longest, (double)(e / 32));
    x.mbytes = s > 1 ? 8e-6 * (double)(BH * rows * s) * D * tensors : 0.0;
  };
  work(blocks);
  add(blocks, splits, each);
  for (int r = 1; r <= (D == 128 ? 2 : 1); ++r) {
    work(r);
    int64_t last = 0;
    for (const int64_t s : counts) {
      if (s > 1 && !parts) break;
      const int64_t e = (tiles + s - 1) / s, real = (tiles + e - 1) / e;
      if (real == last || (real > 1 && (BH * w.blocks * real > 600 || BH * rows * D * tensors * real > MAX_PART_FLOATS))) continue;
      last = real;
      add(r, real, e * 64);
    }
  }
  return found;
}

static void plan_pair(int64_t BH, int64_t Nq, int64_t Nk, int D, bool causal, BwdPlan *p) {
  static const PairCost cost[3][2] = {   // [head_dim 64, 128, 256][causal]
      {{8.73, 0.496, 3.04, 0.196, {2.45, 5.76}, 0.739, {{0.647, 0.649}, {0.324, 0.409}}, 0.333, 0.167},
       {7.42, 0.435, 3.08, 0.162, {7.66, 8.85}, 0.797, {{0.506, 0.491}, {0.324, 0.368}}, 0.508, 0.232}},
      {{8.99, 0.352, 3.34, 0.145, {5.54, 7.33}, 0.646, {{0.814, 1.36}, {0.474, 0.745}}, 0.172, 0.0225},
       {9.07, 0.353, 3.17, 0.145, {8.54, 7.68}, 0.551, {{0.661, 1.09}, {0.451, 0.738}}, 0.184, -0.0585}},
      {{4.44, 0.268, 5.36, 0.139, {9.65, 6.67}, 0.545, {{1.25, 0}, {0.949, 0}}, 0.038, -0.047},
       {4.04, 0.24, 4.86, 0.137, {13.2, 8}, 0.522, {{1.06, 0}, {0.872, 0}}, 0.0869, -0.0534}}};
  const auto two_launches = [](const Share &a, const Share &b) { return a.splits > 1 && b.splits > 1 && 5e5 * (a.mbytes + b.mbytes) > SUM_BETWEEN; };
  // More workgroups are not divided here (96 heads of 691, causal, 94.9 us, took 117.7 with dQ's keys in two parts), but at head_dim 128
  // their rows per wave are chosen together too, by constants fitted to 650 such shapes, none of them divided: they know no cost of
  // parts.  Where queries and keys are within a factor of two and a sixteenth is promised, and up to where it was measured; it takes
  // longer the more workgroups there are.  Against each kind's own choice, in one launch too, over 1128 of the shapes that move: 0.918 of the
  // time without a mask and as many queries as keys, 0.951 with other numbers, causal 0.958, six of them more than 1.04 times (1.065
  // at most); 170 heads of 1056 454 -> 412 us.  Beyond a factor of four 0.965, but one in six more than 1.04 times (53 heads, 415 x 2158:
  // 125 -> 147 us)
  static const PairCost full128[2] = {{8.37, 0.4, 0, 0, {12.2, 3.76}, 0.306, {{0.532, 0.865}, {0.764, 1.12}}, 0, 0.0225},
                                      {7.78, 0.325, 0, 0, {9.93, 7.46}, 0.663, {{0.792, 1.29}, {0.429, 0.613}}, 0, -0.0585}};
  const int64_t wgs = BH * ((Nq + 127) / 128 + (Nk + 127) / 128);
  const bool full = BH > MAX_WGS_BWD || wgs > MAX_WGS_BWD;
  if (full && (D != 128 || wgs > 6000 || 2 * std::min(Nq, Nk) < std::max(Nq, Nk) || p->splits_dkv > 1 || p->splits_dq > 1)) return;
  const PairCost &c = full ? full128[causal] : cost[D == 64 ? 0 : D == 128 ? 1 : 2][causal];
  Share kv[MAX_SHARES], q[MAX_SHARES];
  const int nkv = shares(BH, Nk, Nq, D, causal, false, Nk - Nq, 2, !full, p->blocks_dkv, p->splits_dkv, p->queries_per_split, kv);
  const int nq = shares(BH, Nq, Nk, D, causal, true, Nk - Nq, 1, !full, p->blocks_dq, p->splits_dq, p->keys_per_split, q);
  // (of parts this large each kind fills the chip by itself: 2 heads, 7500 to 8000 of 256, causal, lost 3 to 5 % by the estimate)
  if (kv[0].splits > 1 && q[0].splits > 1 && 5e5 * (kv[0].mbytes + q[0].mbytes) > SUM_BETWEEN * 5 / 8) return;
  const double fixed = c.base + c.prep * 1e-6 * (double)BH * D * (double)(7 * Nq + 3 * Nk);
  double best = (full ? 0.94 : 0.9) * (fixed + pair_time(c, D, kv[0], q[0])) - fixed;
  const Share *bk = &kv[0], *bq = &q[0];
  for (int i = 0; i < nkv; ++i)
    for (int j = 0; j < nq; ++j) {
      const double t = pair_time(c, D, kv[i], q[j]);
      if (t < best && !two_launches(kv[i], q[j])) {
        best = t;
        bk = &kv[i];
        bq = &q[j];
      }
    }
  // Undivided dK / dV of 64 rows per wave beside workgroups of dQ that do not run at once with them: the estimate takes too little where those
  // of 32 rows would all run at once, since half as many take twice as long each and have nothing behind which to hide what is left of
  // dQ.  Of 139 random calls for which 64 rows were chosen ten are such, and they took 1.07 to 1.17 times as long as with 32 (7 heads of
  // 4192: 208 -> 243 us; 0.95 without a mask and with whole tiles of queries, 4224: 205 -> 195); the others 0.898, 1.06 at most
  if (!full && bk != kv && bk->blocks == 2 && bk->splits == 1 && bq->splits == 1 && bk->n + bq->n > 256.0)
    for (int i = 0; i < nkv; ++i)
      if (kv[i].blocks == 1 && kv[i].splits == 1 && kv[i].n <= 256.0) bk = &kv[i];
  p->blocks_dkv = bk->blocks; p->splits_dkv = bk->splits; p->queries_per_split = bk->each;
  p->blocks_dq = bq->blocks; p->splits_dq = bq->splits; p->keys_per_split = bq->each;
}

BwdPlan bwd_plan(int64_t BH, int64_t Nq, int64_t Nk, int D, int causal, int may_split) {
  // [head_dim][32-row blocks per wave], in tiles of 32 rows
  static const SplitCost dkv64[2] = {{{0.522, 0.590, 0}, 2, 0.462, 0.662, 2.96, 0.186, 0}, {}},
                         dkv128[2] = {{{0.642, 0, 0}, 1, 0.373, 0.541, 3.96, 0.174, 0}, {{0.756, 0, 0}, 1, 0.373, 0.541, 3.96, 0.174, 0}},
                         dkv256[2] = {{{1.137, 0, 0}, 1, 3.005, 0.686, 7.39, 0.143, 0}, {}},
                         dq64[2] = {{{0.337, 0.473, 0}, 2, 0.255, 0.515, 2.74, 0.254, 0}, {}},
                         dq128[2] = {{{0.448, 0, 0}, 1, 0.577, 0.585, 3.62, 0.245, 0}, {{0.668, 0, 0}, 1, 0.577, 0.585, 3.62, 0.245, 0}},
                         dq256[2] = {{{0.852, 0, 0}, 1, 3.596, 0.833, 4.97, 0.147, 0}, {}};
  const float f = (float)Nq / (float)Nk;
  BwdPlan p;
  bwd_part(BH, Nk, Nq, D, causal, false, Nk - Nq, f, may_split, D == 64 ? dkv64 : D == 128 ? dkv128 : dkv256, 2, &p.blocks_dkv,
           &p.splits_dkv, &p.queries_per_split);
  bwd_part(BH, Nq, Nk, D, causal, true, Nk - Nq, f, may_split, D == 64 ? dq64 : D == 128 ? dq128 : dq256, 1, &p.blocks_dq, &p.splits_dq,
           &p.keys_per_split);
  if (may_split) plan_pair(BH, Nq, Nk, D, causal != 0, &p);
  const int64_t kv = p.splits_dkv > 1 ? BH * D * 8 * Nk * p.splits_dkv : 0, q = p.splits_dq > 1 ? BH * D * 4 * Nq * p.splits_dq : 0;
  // large parts of both: dK and dV are added before dQ starts, whose parts take their place.  One launch more, of a call of
  // milliseconds (2 heads, 16384 x 16384 of 256, causal, forward and backward: 1939 -> 1908 us); smaller ones lose by it (4 heads of
  // 2300: 188 -> 191)
  // (and what one launch of 2^32 - 1 threads does not hold: 8388607 heads, whose staging launch is not too large)
  const auto wgs = [&](int64_t rows, int blocks, int splits) { return (BH * ((rows + 128 * blocks - 1) / (128 * blocks)) + 7) / 8 * 8 * splits; };
  p.sum_between = (kv > 0 && q > 0 && kv + q > SUM_BETWEEN) ||
                  wgs(Nk, p.blocks_dkv, p.splits_dkv) + wgs(Nq, p.blocks_dq, p.splits_dq) > 0xffffffffLL / 256;
  p.part_bytes = p.sum_between ? std::max(kv, q) : kv + q;
  return p;
}

BwdPlan bwd_plan_within(int64_t BH, int64_t Nq, int64_t Nk, int D, int causal, int64_t room) {
  const BwdPlan p = bwd_plan(BH, Nq, Nk, D, causal, 1);
  return p.part_bytes <= room ? p : bwd_plan(BH, Nq, Nk, D, causal, 0);
}

int64_t bwd_split_bytes(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int D, int causal) {
  return bwd_plan(B * H, Nq, Nk, D, causal, 1).part_bytes;
}

}  // namespace qfa
