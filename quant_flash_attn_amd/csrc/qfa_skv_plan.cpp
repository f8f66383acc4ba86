// Which shared-KV kernel takes a call and how its keys are split over workgroups: pure functions of the sizes.
//
// A launch of n workgroups is estimated as rounds of the workgroups that are resident at once; a workgroup costs its tiles and
// `start` once, times what they take on the busiest CU: `alone` and `start` with one workgroup on it, `each` and `start_each` times
// their number with more.  A split adds the launch that merges (`merge` and `per_mb` for every 10^6 floats of partial results).
//
// Forward, and dQ of 256: n is eight times the workgroups of the XCD that gets most (XcdBlock in qfa_skv_common.h deals whole heads).
// 81 heads of three workgroups are 33 on one XCD of 32 CUs, two rounds, where an even deal of 243 would be one: 173 queries,
// 513 keys of 256 took 45.9 us instead of 31.2 while they were counted evenly.  Constants in microseconds, fitted to 5000 shapes of 1
// to 2000 heads, 17 to 512 queries (1024 at head_dim 256) and 64 to 16000 keys, each timed with all kernels and several splits (3 to
// 7 % rms): what they choose takes 1.002 to 1.009 times the best measured choice in the geometric mean, and more than 1.05 times
// what the 16-query kernels take in 0 to 4 of 1700 shapes each.
// The others count evenly, as their constants were fitted (one-pass backward 650 launches each, 5 to 8 % rms, dQ 2 to 4 %): fitted as
// above they made the backward of 700 shapes of 64 and 128 a hundredth slower.
#include <algorithm>

#include "qfa_host.h"
#include "qfa_merge.h"

namespace qfa {
namespace {

struct Cost {
  float base, alone, each, start, start_each, merge, per_mb;
  int resident;   // workgroups per CU
  float of(int64_t n, float tiles, int64_t splits, int64_t partials) const {
    const int64_t slots = 256 * resident, full = n / slots, rem = n % slots;
    const auto round = [&](int64_t c) { return std::max(alone * tiles + start, (each * tiles + start_each) * (float)c); };
    const float rounds = (float)full * round(resident) + (rem ? round((rem + 255) / 256) : 0.0f);
    return base + rounds + (splits > 1 ? merge + per_mb * 1e-6f * (float)partials : 0.0f);
  }
};
// what n is for per_bh workgroups of each of BH heads
enum class Count { Even, Xcd };
int64_t count(Count c, int64_t BH, int64_t per_bh) { return c == Count::Even ? BH * per_bh : xcd_grid(BH, per_bh); }
int by_dim(int D) { return D == 256 ? 2 : D == 128 ? 1 : 0; }

//                               head_dim 64                              128                                      256
// 16 queries per workgroup, tiles of 32 keys dealt to four waves
const Cost kFwd16[3] = {{3.6f, .639f, .361f, .34f, .56f, 2.9f, 2.3f, 3}, {3.9f, .890f, .556f, .84f, 1.05f, 2.8f, 1.9f, 3}, {4.0f, 1.387f, .957f, 2.49f, 2.51f, 3.1f, 1.3f, 2}};
// 32 queries per wave, tiles of 64 keys; two and four waves side by side.  (Four at 256 are faster since their codes are requested a
// tile earlier: fitted again, 2.07 and 8.9, they would take calls at 0.89 of the time in the mean.  Not done: those calls would have
// one reference maximum per query instead of two or four, and an fp16 error against 64 bits 1.0004 to 1.08 times as large, most at
// few keys.)
const Cost kFwdTile[2][3] = {
    {{4.6f, .673f, .377f, .52f, 1.12f, 2.5f, 1.7f, 3}, {2.9f, .870f, .600f, 3.88f, 2.61f, 1.9f, 2.3f, 2}, {1.6f, 1.507f, 0.f, 8.67f, 0.f, 1.1f, 2.5f, 1}},
    {{4.5f, .934f, .607f, .50f, 1.15f, 2.7f, 1.9f, 3}, {3.4f, 1.183f, .908f, 2.64f, 2.50f, 2.5f, 2.4f, 2}, {0.2f, 2.467f, 0.f, 8.17f, 0.f, 2.1f, 2.6f, 1}}};
// one-pass backward: up to 16 queries, up to 32 (650 launches each of 1 to 1500 heads, 300 to 24000 keys, 5 to 8 % rms)
const Cost kPass[2][3] = {
    {{6.1f, 1.638f, 1.159f, .74f, .52f, 2.7f, 2.4f, 2}, {6.0f, 2.717f, 2.163f, 3.18f, 2.53f, 1.8f, 1.5f, 2}, {2.2f, 5.371f, 4.535f, 13.27f, 11.20f, 0.6f, 1.7f, 1}},
    {{4.6f, 1.898f, 1.309f, 2.54f, 1.75f, 2.6f, 1.9f, 2}, {6.6f, 3.010f, 2.324f, 3.07f, 2.37f, 1.7f, 1.6f, 2}, {0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 0.f, 1}}};
// dQ: 16 queries per workgroup; tiles with two and four waves side by side (only their differences matter: no base at 64 and 128)
const Cost kDq16[3] = {{0.f, .602f, .356f, .58f, .35f, 0.f, 0.f, 3}, {0.f, .810f, .664f, .32f, .26f, 0.f, 0.f, 3}, {5.6f, 1.268f, .941f, 2.86f, 2.90f, 0.f, 0.f, 2}};
const Cost kDqTile[2][3] = {
    {{0.f, .998f, .548f, 0.f, 0.f, 2.7f, 1.8f, 3}, {0.f, 1.336f, .932f, .28f, .20f, 2.4f, 2.0f, 2}, {5.2f, 2.728f, 0.f, 6.42f, 0.f, 2.9f, 1.9f, 1}},
    {{0.f, 1.284f, .482f, 0.f, 0.f, 4.0f, 1.9f, 3}, {0.f, 2.015f, 1.326f, 0.f, 0.f, 3.8f, 1.7f, 2}, {5.2f, 3.763f, 0.f, 5.22f, 0.f, 5.1f, 1.5f, 1}}};

const int kSplits[] = {1, 2, 3, 4, 6, 8, 12, 16, 24, 32, 48, 64};

// The best split of `tiles` tiles for per_bh workgroups of each head; at least two tiles each, partial results of at most `room` floats.
// Only a cost below `limit` matters to the caller: no split is looked at where the merge and two tiles already take that long (most
// small calls, whose 10 us this function is part of)
void best_split(const Cost &c, Count how, int64_t BH, int64_t per_bh, int64_t rows, int64_t tiles, float per, int64_t row_floats,
                int64_t room, float limit, int *splits, int64_t *tiles_each, float *cost) {
  *splits = 1;
  *cost = 3e38f;
  for (const int s : kSplits) {
    if (s > 1 && (2 * s > tiles || BH * per_bh * s > 1600 || rows * s * row_floats > room)) break;
    if (s > 1 && c.base + (c.alone * (per * 2.0f) + c.start) + c.merge >= limit) break;
    const int64_t each = (tiles + s - 1) / s, used = (tiles + each - 1) / each;
    const float t = c.of(count(how, BH, per_bh * used), per * (float)each, used, rows * used * row_floats);
    if (t < (s > 1 && *splits == 1 ? 0.9f : 1.0f) * *cost) {   // (a split has to promise a tenth)
      *cost = t;
      *splits = (int)used;
      *tiles_each = each;
    }
  }
}
// two or four waves side by side on the queries, the keys split
SkvTilePlan best_tile(const Cost (*c)[3], Count how, int64_t BH, int64_t Nq, int64_t Nk, int D, int64_t row_floats, int64_t room, float limit,
                      float *cost) {
  const int64_t blocks = (Nq + 31) / 32, tiles = (Nk + 63) / 64;
  SkvTilePlan p = {2, 1, (int)tiles};
  *cost = 3e38f;
  for (int i = 0; i < (blocks > 2 ? 2 : 1); ++i) {
    const int qw = i ? 4 : 2;
    int splits = 1;
    int64_t each = tiles;
    float t;
    best_split(c[i][by_dim(D)], how, BH, (blocks + qw - 1) / qw, BH * Nq, tiles, 1.0f, row_floats, room, std::min(limit, *cost), &splits, &each, &t);
    if (t < *cost) {
      *cost = t;
      p = {qw, splits, (int)each};
    }
  }
  return p;
}

// the 16-query kernel
void fwd16_plan(int64_t BH, int64_t Nq, int64_t Nk, int D, int *splits, int *tiles_per_split) {
  // as many workgroups as are resident at once (three per CU; a second, partly filled round costs a whole one), at head_dim
  // 256 about four per CU (two are resident), or what split_plan finds better
  const int64_t wgs = BH * ((Nq + 15) / 16);
  const int64_t fill = D == 256 ? (wgs >= 512 ? 1 : (1024 + wgs - 1) / wgs) : 768 / wgs;
  const int64_t ntiles = (Nk + 31) / 32, rows = BH * Nq;
  split_plan(wgs, rows, ntiles, D, fill, splits, tiles_per_split);
  // Blocks of more than 16 queries that the tile kernels could take keep within the built-in scratch, as those do: which of the two
  // is chosen does not decide whether a call without a workspace of its own is accepted
  if (Nq > 16 && *splits > 1 && split_partial_bytes(rows, *splits, D) > QFA_STATIC_SCRATCH_BYTES) {
    const int64_t most = std::max<int64_t>(1, QFA_STATIC_SCRATCH_BYTES / split_partial_bytes(rows, 1, D));
    const int64_t each = (ntiles + most - 1) / most;
    *tiles_per_split = (int)each;
    *splits = (int)((ntiles + each - 1) / each);
  }
}

}  // namespace

SkvFwdPlan skv_fwd_plan(int64_t BH, int64_t Nq, int64_t Nk, int D) {
  SkvFwdPlan f = {{0, 1, 0}, 1, 0, 0};
  fwd16_plan(BH, Nq, Nk, D, &f.splits, &f.tiles_per_split);
  if (Nq > 16) {
    const float t16 = kFwd16[by_dim(D)].of(count(Count::Xcd, BH, (Nq + 15) / 16 * f.splits), 0.25f * (float)f.tiles_per_split, f.splits,
                                           BH * Nq * f.splits * (D + 2));
    // (with 32 queries or fewer half of the waves have none)
    const float limit = (Nq <= 32 ? 0.85f : 0.93f) * t16;
    // (partial results within the built-in scratch at every head_dim)
    float t;
    const SkvTilePlan p = best_tile(kFwdTile, Count::Xcd, BH, Nq, Nk, D, D + 2, QFA_STATIC_SCRATCH_BYTES / 4, limit, &t);
    if (t < limit) f.tile = p;
  }
  const int parts = f.tile.qw ? f.tile.splits : f.splits;
  f.part_bytes = parts > 1 ? split_partial_bytes(BH * Nq, parts, D) : 0;
  return f;
}

SkvTilePlan skv_tile_dq_plan(int64_t BH, int64_t Nq, int64_t Nk, int D) {
  const Count how = D == 256 ? Count::Xcd : Count::Even;
  const float t16 = kDq16[by_dim(D)].of(count(how, BH, (Nq + 15) / 16), 0.25f * (float)((Nk + 31) / 32), 1, 0);
  // (33 to 48 queries leave a quarter of two waves' work to padding: 1024 heads, 48 queries, 3000 keys of 128 take 178 us with
  // the one kernel and 208 with the other)
  const float limit = (Nq > 48 ? 0.93f : D == 256 ? 0.85f : 0.75f) * t16;
  float t;
  const SkvTilePlan p = best_tile(kDqTile, how, BH, Nq, Nk, D, D, 16 << 20, limit, &t);
  return t < limit ? p : SkvTilePlan{0, 1, 0};
}

// One workgroup per (batch, head) does the whole backward, one on a CU at head_dim 128 and two at 64, and leaves the head's keys
// unsplit.  Timed beside the two kernels with their splits in 29000 calls of 48 to 6000 heads, 33 to 128 queries and 16 to 65000 keys,
// it takes 0.79 (head_dim 64) and 0.73 (128) of their time in the mean of what it is given.  Left out:
//   few heads over long keys, which the others split (95 heads, 117 x 8400 of 64: 308 against 146 us), and with them all calls of
//     fewer than 320 heads of 64 and 128 of 128, where it would be faster up to about 1500 keys (151 heads, 128 x 24: 7 against 18);
//   257 to 287 heads of 128, a second round of a few heads: 1.02 to 1.06 over long keys;
//   thousands of heads of 128 with one or two tiles each: its start weighs more than theirs (1.02).
// Over long keys 320 to 699 heads of 64 and 128 to 329 of 128 leave a round nearly empty or the first one half full, and which is faster
// depends on the queries too: there both are estimated.
namespace {
// us of the pass: start, a tile, a tile of 1000 heads (the clock falls with the CUs at work; with more than 96 queries `wave4` more), and
// the second round, its tiles and its start, where there are more heads than workgroups at once
struct PassCost { float start, tile, heads, wave4, tile2, start2; };
// of the two kernels, in proportion to 1000 heads but for the start: a tile, that for every 16 queries, every 32, a head, and what a tile
// takes less with at most 48 queries (the 16-query kernel forms dQ)
struct TwoCost { float start, tile, q16, q32, head, few; };
// Fitted to 3900 calls of 64 and 4000 of 128, 1500 to 65000 keys (3 % rms, the two kernels 5).  What it chooses takes 1.003 (64) and 1.000
// (128) times the better one in the mean of 9000 such calls, more than 1.04 times in 136 and 12, 1.11 at most; the pass always 1.008 and
// 1.001, 360 and 54, 1.21; edges in heads and keys alone 1.014 and 1.012, 654 and 396, 1.38 (297 heads, 116 x 2560 of 128: 290, 210 us)
const PassCost kPassHead[2][2] = {{{3.7f, 1.693f, 1.133f, 0.f, 1.467f, -4.2f}, {4.1f, 2.461f, 1.544f, .484f, 1.635f, 3.1f}},
                                  {{0.9f, 1.283f, 2.816f, 0.f, 1.222f, 5.5f}, {7.3f, 1.705f, 3.374f, .463f, 1.772f, 8.5f}}};
const TwoCost kTwo[2] = {{21.6f, 3.032f, .085f, 1.487f, -0.7f, .433f}, {35.5f, 5.198f, .478f, 2.281f, -5.1f, .834f}};
bool pass_pays(int64_t BH, int64_t Nq, int64_t Nk, int D) {
  const PassCost &p = kPassHead[by_dim(D)][Nq > 64];
  const TwoCost &w = kTwo[by_dim(D)];
  const float tiles = (float)((Nk + 63) / 64), heads = 1e-3f * (float)BH;
  const float pass = p.start + tiles * (p.tile + heads * (p.heads + (Nq > 96 ? p.wave4 : 0.f))) + (BH > (D == 64 ? 512 : 256) ? p.start2 + p.tile2 * tiles : 0.f);
  const float two = w.start + heads * (w.head + tiles * (w.tile - (Nq <= 48 ? w.few : 0.f) + w.q16 * (float)((Nq + 15) / 16) + w.q32 * (float)((Nq + 31) / 32)));
  return pass <= 1.01f * two;
}
enum class Pass { No, Estimate, Yes };
Pass pass_of(int64_t BH, int64_t Nq, int64_t Nk, int D) {
  if (Nq <= 32 || Nq > 128 || BH > 0x7fffffffLL) return Pass::No;
  if (D == 64) return BH < 320 ? Pass::No : BH < 700 && Nk >= 1500 ? Pass::Estimate : Pass::Yes;
  if (D != 128 || BH < 128 || (BH > 256 && BH < 288)) return Pass::No;
  if (BH < 330) return Nk >= 1500 ? Pass::Estimate : Pass::Yes;
  return Nk > 128 || BH <= 1024 ? Pass::Yes : Pass::No;
}
}  // namespace

bool skv_pass_takes(int64_t BH, int64_t Nq, int64_t Nk, int D) {
  const Pass p = pass_of(BH, Nq, Nk, D);
  return p == Pass::Yes || (p == Pass::Estimate && pass_pays(BH, Nq, Nk, D));
}
// Without scratch dQ's keys are not split either: what the estimate gives to a split goes to the pass then (87 such calls: 0.97 of the time
// of the two kernels in the mean, 0.84 to 1.10; 355 heads, 85 x 13075 of 64: 622 us, with scratch 603, without 732)
bool skv_pass_takes_unsplit(int64_t BH, int64_t Nq, int64_t Nk, int D) {
  return skv_pass_takes(BH, Nq, Nk, D) || (pass_of(BH, Nq, Nk, D) == Pass::Estimate && skv_tile_dq_plan(BH, Nq, Nk, D).splits > 1);
}

int skv_bwd_splits(int64_t BH, int64_t Nq, int64_t Nk, int D) {
  int splits = 1;
  int64_t each;
  float t;
  best_split(kPass[Nq <= 16 ? 0 : 1][by_dim(D)], Count::Even, BH, 1, BH * Nq, (Nk + 31) / 32, 0.25f, D, 16 << 20, 3e38f, &splits, &each, &t);
  return splits;
}

int64_t skv_bwd_workspace_bytes(int64_t B, int64_t H, int64_t Nq, int64_t Nk, int D) {
  // The one pass needs none.  Where a layout with the heads inside the tokens would not fit it (skv_pass_fits; the strides are not known
  // here) the answer is what the two kernels want; still wider strides run without.
  if (skv_pass_takes(B * H, Nq, Nk, D) && skv_pass_fits(Nk, H * D, H * D, H * D)) return 0;
  const int s = skv_bwd_one_pass(Nq, D) ? skv_bwd_splits(B * H, Nq, Nk, D) : skv_tile_dq_plan(B * H, Nq, Nk, D).splits;
  return s > 1 ? B * H * Nq * s * (int64_t)D * 4 : 0;
}

}  // namespace qfa
